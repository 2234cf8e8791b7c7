"""The first two iterations of 11 x 11 and 9 x 9 windows take workgroup tiles of half
the height where that evens out the CUs: a view's results are the bits of the batched form's on
both sides of the rule, with ragged tiles."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# W, H, S; tiles of 64 x 8 pixels and of 64 x 4
CASES = [
    (640, 480, 2),   # 600 or 1200: halves
    (599, 449, 2),   # 570 or 1130, ragged both ways: halves
    (480, 360, 1),   # 360 or 720: halves
    (561, 421, 2),   # 477 or 954: not
    (680, 510, 2),   # 704 or 1408: not
]


@pytest.mark.parametrize("W,H,S", CASES)
@pytest.mark.parametrize("radius,store", [(5, 0), (5, 1), (4, 0), (4, 1)])
def test_view_equals_batched_view(pkg, ctx, scenes, W, H, S, radius, store):
    job = scenes.sphere_job(W, H, S, scene_seed=W + S, radius=radius, stride=1)
    hs = [ctx.upload(im, store) for im in [job.ref] + job.srcs]
    try:
        desc = pkg.make_desc(hs[0], hs[1:], job.Kinv, job.A, job.b, job.dmin, job.dmax,
                             radius=radius, stride=1, iterations=3, seed=W * H)
        one = ctx.run_view(desc, (H, W))
        many = ctx.batch_run([desc], [(H, W)])[0]
        for k in ("depth", "normal", "cost"):
            assert np.array_equal(one[k], many[k]), k
    finally:
        for h in hs:
            ctx.release(h)
