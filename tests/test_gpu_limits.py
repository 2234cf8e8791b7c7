"""Calls at the limits of device memory: what fits is accepted, and a request that
was refused leaves nothing behind for the next call."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOO_MUCH = 1 << 45   # more than the card has, within the context's own budget


def test_a_refused_allocation_is_not_reported_again(pkg, scenes):
    job = scenes.plane_job(W=160, H=120, iterations=1)
    with pkg.Context(hbm_budget=1 << 50) as c:
        hs = [c.upload(im) for im in [job.ref] + job.srcs]
        desc = pkg.make_desc(hs[0], hs[1:], job.Kinv, job.A, job.b, job.dmin, job.dmax,
                             iterations=1, seed=3)
        want = c.run_view(desc, job.shape)
        with pytest.raises(pkg.HP3DError):
            c.device_alloc(TOO_MUCH)
        got = c.run_view(desc, job.shape)
        for k in ("depth", "normal", "cost"):
            assert np.array_equal(got[k], want[k]), k
        with pytest.raises(pkg.HP3DError):
            pkg.Server(TOO_MUCH, max_jobs=2)
        assert np.array_equal(c.run_view(desc, job.shape)["depth"], want["depth"])


def small_views(n, W=40, H=30):
    rng = np.random.default_rng(n)
    K = np.array([[36.0, 0, W / 2], [0, 36.0, H / 2], [0, 0, 1.0]])
    maps = []
    for k in range(n):
        d = rng.uniform(1, 5, (H, W)).astype(np.float32)
        d[rng.random((H, W)) < 0.4] = 0
        maps.append(dict(depth=d, confidence=rng.random((H, W)).astype(np.float32),
                         normal=rng.normal(size=(H, W, 3)).astype(np.float32),
                         color=rng.integers(0, 256, (H, W), dtype=np.uint8), K=K, R=np.eye(3),
                         t=np.array([0.1 * k, 0, 0])))
    return maps


@pytest.mark.parametrize("n,W,H", [(1, 40, 30), (40, 40, 30), (12, 300, 200), (3, 1, 1)])
def test_fusion_in_the_memory_that_one_view_at_a_time_needs(pkg, orc, n, W, H):
    """The maps, the output, and the counts and offsets of 256-pixel blocks of the
    largest view are enough, however many views there are."""
    maps = small_views(n, W, H)
    maps[0]["depth"][0, 0], maps[0]["confidence"][0, 0] = 2.0, 1.0
    want = orc.fuse(maps, min_confidence=0.3)

    def a256(b):
        return (b + 255) // 256 * 256

    px = W * H
    blocks = (px + 255) // 256
    need = n * (2 * a256(4 * px) + a256(12 * px) + a256(px))
    need += a256(4 * blocks) + a256(8 * blocks) + 256 + 36 * len(want[0])
    with pkg.Context(hbm_budget=need) as c:
        for _ in range(2):
            for g, w in zip(c.fuse(maps, min_confidence=0.3), want):
                assert np.array_equal(g, w)
