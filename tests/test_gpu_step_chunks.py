"""A step of many views gives every XCD chunks of 16, 32 or 64 tiles, by the
step's tile count and the storage: each view's results are the bits of its own
per-view solve on both sides of each line, with a ragged last chunk, and with
views that leave the step before the others."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("store", [0, 1])
@pytest.mark.parametrize("copies", [1, 3, 4, 7])     # 602, 1806, 2408 and 4214 tiles a step
def test_views_of_a_step_equal_their_own_solve(pkg, ctx, scenes, store, copies):
    W, H, S = 641, 479, 2
    job = scenes.sphere_job(W, H, S, scene_seed=9, radius=2, stride=1)
    hs = [ctx.upload(im, store) for im in [job.ref] + job.srcs]
    try:
        descs = [pkg.make_desc(hs[0], hs[1:], job.Kinv, job.A, job.b, job.dmin, job.dmax,
                               radius=2, stride=1, iterations=1 + (k == 0), seed=100 + k)
                 for k in range(copies)]
        outs = ctx.batch_run(descs, [(H, W)] * copies)
        for d, o in zip(descs, outs):
            one = ctx.run_view(d, (H, W))
            for key in ("depth", "normal", "cost"):
                assert np.array_equal(one[key], o[key]), key
    finally:
        for h in hs:
            ctx.release(h)
