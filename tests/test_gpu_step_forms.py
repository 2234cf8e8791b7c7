"""Steps of 7 x 7 windows have an instance for START items alone beside the plain
and the pooled one: views that end at their START, after one and after several
iterations give the bits of their own per-view solve, in steps below and above the
pooled form's 1024 tiles."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("store", [0, 1])
@pytest.mark.parametrize("W,H,copies", [(161, 97, 1), (161, 97, 3), (641, 479, 2)])  # 42 to 1260 tiles
def test_views_of_every_length(pkg, ctx, scenes, store, W, H, copies):
    job = scenes.sphere_job(W, H, 2, scene_seed=W, radius=3, stride=1)
    hs = [ctx.upload(im, store) for im in [job.ref] + job.srcs]
    try:
        for iterations in ([0] * copies, list(range(copies)), [2] + [0] * (copies - 1)):
            descs = [pkg.make_desc(hs[0], hs[1:], job.Kinv, job.A, job.b, job.dmin, job.dmax,
                                   radius=3, stride=1, iterations=n, seed=7 + k)
                     for k, n in enumerate(iterations)]
            outs = ctx.batch_run(descs, [(H, W)] * copies)
            for d, o in zip(descs, outs):
                one = ctx.run_view(d, (H, W))
                for key in ("depth", "normal", "cost"):
                    assert np.array_equal(one[key], o[key]), (iterations, key)
    finally:
        for h in hs:
            ctx.release(h)
