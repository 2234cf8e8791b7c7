"""Views of few pixels: the per-view entry point splits a pixel's evaluations
over a workgroup's waves, the batched form evaluates them in one lane.  Their
results are the same bits, on both sides of every line of the split rule
(tiles of 32 x 4 pixels, sources, taps), ragged tiles and every wave count
among them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# W, H, S, radius, stride, store, top_k, iterations
CASES = [
    (17, 13, 1, 5, 1, 0, 3, 2),      # one ragged tile column, one source
    (33, 31, 2, 5, 2, 1, 1, 3),      # 8 waves, both steps side by side
    (96, 72, 3, 2, 1, 0, 2, 3),
    (96, 72, 5, 5, 1, 0, 3, 2),      # 15 waves
    (97, 71, 8, 4, 2, 1, 8, 3),      # 16 waves, 24 evaluations for the two steps
    (161, 127, 6, 1, 1, 0, 4, 3),    # 8 waves
    (255, 163, 4, 3, 1, 1, 3, 2),    # 4 waves
    (320, 240, 1, 5, 1, 0, 3, 2),    # 600 tiles, S = 1: split above 49 taps ...
    (320, 240, 1, 5, 2, 0, 3, 2),    # ... and not below
    (352, 284, 2, 5, 2, 0, 3, 2),    # 781 of 800 tiles: split
    (352, 300, 2, 5, 2, 0, 3, 2),    # 825: not
    (640, 75, 2, 5, 1, 0, 3, 2),     # the initial cost's line is further out
    (641, 479, 1, 3, 1, 0, 3, 1),    # neither is split
]


@pytest.mark.parametrize("W,H,S,radius,stride,store,top_k,iterations", CASES)
def test_split_view_equals_batched_view(pkg, ctx, scenes, W, H, S, radius, stride, store, top_k,
                                        iterations):
    job = scenes.sphere_job(W, H, S, scene_seed=W + S, radius=radius, stride=stride)
    hs = [ctx.upload(im, store) for im in [job.ref] + job.srcs]
    try:
        desc = pkg.make_desc(hs[0], hs[1:], job.Kinv, job.A, job.b, job.dmin, job.dmax,
                             radius=radius, stride=stride, iterations=iterations, top_k=top_k,
                             seed=W * H + S)
        one = ctx.run_view(desc, (H, W))
        many = ctx.batch_run([desc], [(H, W)])[0]
        for k in ("depth", "normal", "cost"):
            assert np.array_equal(one[k], many[k]), k
        # the initial cost by itself, and of given hypotheses
        d0, n0 = ctx.init_hypotheses(desc, (H, W))
        desc.iterations = 0
        assert np.array_equal(ctx.run_view(desc, (H, W))["cost"], ctx.cost_eval(desc, d0, n0))
        assert np.array_equal(ctx.batch_run([desc], [(H, W)])[0]["cost"],
                              ctx.cost_eval(desc, d0, n0))
    finally:
        for h in hs:
            ctx.release(h)
