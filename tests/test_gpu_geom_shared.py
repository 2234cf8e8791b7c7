"""The geometric filter's counts where views share host memory: of the maps as they are
when the call returns, whose bytes are those of the later view."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shared", ["depth", "confidence is depth", "nothing"])
def test_counts_of_maps_that_share_memory(pkg, ctx, shared):
    W, H = 97, 41
    rng = np.random.default_rng(11)
    K = np.array([[90.0, 0, W / 2], [0, 90.0, H / 2], [0, 0, 1.0]])
    maps = []
    for v in range(4):
        d = (3.0 + 0.6 * rng.random((H, W))).astype(np.float32)
        d[rng.random((H, W)) < 0.2] = 0
        maps.append(dict(depth=d, normal=np.zeros((H, W, 3), np.float32), K=K, R=np.eye(3),
                         t=np.array([0.02 * v, 0, 0]), src=[u for u in range(4) if u != v]))
    if shared == "depth":
        maps[2]["depth"] = maps[0]["depth"]
        maps[2]["src"] = [1, 3]
    elif shared == "confidence is depth":
        maps[3]["confidence"] = maps[1]["depth"]
    kept = ctx.geom_filter(maps, depth_tol=0.05, min_consistent=2)
    assert kept == [int((m["depth"] > 0).sum()) for m in maps]
    if shared == "depth":
        assert kept[0] == kept[2]
