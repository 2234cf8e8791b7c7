"""Fusion over blocks of 2048 pixels: views around a block's edges, of different
sizes, with every map present or absent, ranked as the oracle ranks them; and
the filter's counts of pixels left."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def a_map(rng, W, H, conf, normal, color):
    K = np.array([[0.9 * W, 0, W / 2], [0, 0.9 * W, H / 2], [0, 0, 1.0]])
    th = rng.uniform(-0.3, 0.3)
    R = np.array([[np.cos(th), 0, np.sin(th)], [0, 1, 0], [-np.sin(th), 0, np.cos(th)]])
    d = rng.uniform(1, 5, (H, W)).astype(np.float32)
    d[rng.random((H, W)) < 0.4] = 0
    m = dict(depth=d, K=K, R=R, t=rng.normal(size=3))
    if conf:
        m["confidence"] = rng.random((H, W)).astype(np.float32)
    if normal:
        m["normal"] = rng.normal(size=(H, W, 3)).astype(np.float32)
    if color:
        m["color"] = rng.integers(0, 256, (H, W) + ((3,) if color == 3 else ()), dtype=np.uint8)
    return m


@pytest.mark.parametrize("sizes", [
    [(1, 1)], [(2047, 1)], [(64, 32)], [(2049, 1)], [(45, 91), (1, 1), (64, 32)],
    [(333, 77), (2048, 2), (31, 17), (640, 480)],
])
def test_blocks(pkg, orc, ctx, sizes):
    rng = np.random.default_rng(len(sizes) * 1000 + sizes[0][0])
    maps = [a_map(rng, W, H, k % 2 == 0, k % 3 != 1, (1, 3, 0)[k % 3])
            for k, (W, H) in enumerate(sizes)]
    maps[0]["depth"][0, 0] = 2.0
    got = ctx.fuse(maps, min_confidence=0.3)
    want = orc.fuse(maps, min_confidence=0.3)
    for g, w in zip(got, want):
        assert np.array_equal(g, w)
    only = ctx.fuse(maps, min_confidence=0.3, with_normals=False, with_colors=False)
    assert np.array_equal(only[0], want[0]) and only[1] is None and only[2] is None


@pytest.mark.parametrize("W,H", [(64, 4), (65, 5), (203, 61), (17, 301)])
def test_filter_counts_what_it_leaves(pkg, ctx, W, H):
    rng = np.random.default_rng(W)
    maps = []
    for v in range(4):
        m = a_map(rng, W, H, v != 2, True, 0)
        m["depth"] = (3.0 + 0.6 * rng.random((H, W))).astype(np.float32)
        m["depth"][rng.random((H, W)) < 0.2] = 0
        m.update(R=np.eye(3), t=np.array([0.01 * v, 0, 0]), src=[u for u in range(4) if u != v])
        maps.append(m)
    maps[3]["src"] = [0]                 # fewer sources than asked for: left as it is
    before = maps[3]["depth"].copy()
    kept = ctx.geom_filter(maps, depth_tol=0.05, min_consistent=2)
    assert kept[3] == -1 and np.array_equal(maps[3]["depth"], before)
    assert kept[:3] == [int((m["depth"] > 0).sum()) for m in maps[:3]]
    assert 0 < min(kept[:3]) < W * H
