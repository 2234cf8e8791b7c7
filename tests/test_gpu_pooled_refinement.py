"""The pooled form of the refinement (early iterations, views and steps of many
tiles) gives the bits of the plain form: a view of 845 tiles is pooled in the
per-view form and not in a step by itself, nor at strides 2; two of them in one
step are.  Source counts and means on both sides of the rule, ragged tiles,
iterations across its last pooled one, and images of no texture, whose costs
are all equal."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# S, radius, stride, store, top_k, iterations
CASES = [
    (2, 5, 1, 0, 3, 2),
    (2, 3, 1, 1, 2, 8),      # the last two iterations are plain again
    (3, 2, 1, 0, 3, 3),      # 5 taps: plain in either
    (4, 5, 2, 0, 3, 2),
    (5, 5, 2, 1, 2, 3),
    (8, 4, 1, 0, 3, 2),
    (4, 4, 1, 1, 8, 2),      # a mean over more than three: plain
    (3, 5, 1, 0, 1, 2),      # over one: plain
    (1, 5, 1, 0, 3, 2),      # one source: plain
]


@pytest.mark.parametrize("flat", [False, True])
@pytest.mark.parametrize("S,radius,stride,store,top_k,iterations", CASES)
def test_pooled_equals_plain(pkg, ctx, scenes, S, radius, stride, store, top_k, iterations, flat):
    W, H = 799, 519
    job = scenes.sphere_job(W, H, S, scene_seed=3 + S, radius=radius, stride=stride)
    images = [job.ref] + job.srcs
    if flat:
        images = [np.full_like(im, 90) for im in images]
        images[0][100:300, 200:500] = job.ref[100:300, 200:500]
    hs = [ctx.upload(im, store) for im in images]
    try:
        def desc(seed):
            return pkg.make_desc(hs[0], hs[1:], job.Kinv, job.A, job.b, job.dmin, job.dmax,
                                 radius=radius, stride=stride, iterations=iterations, top_k=top_k,
                                 seed=seed)
        d = desc(11)
        one = ctx.run_view(d, (H, W))
        outs = ctx.batch_run([d], [(H, W)])
        outs.append(ctx.batch_run([d, desc(12)], [(H, W)] * 2)[0])
        for o in outs:
            for key in ("depth", "normal", "cost"):
                assert np.array_equal(one[key], o[key]), key
    finally:
        for h in hs:
            ctx.release(h)
