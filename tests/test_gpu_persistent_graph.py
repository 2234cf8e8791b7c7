"""A persistent batch replays its graph only for the schedule it was captured with: the
same views with other iteration counts, one after another, each equal their own
per-view solve bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_iteration_counts_change_between_batches(pkg, scenes):
    job = scenes.sphere_job(161, 97, 2, scene_seed=3, radius=2, stride=1)
    with pkg.Context() as c:
        hs = [c.upload(im) for im in [job.ref] + job.srcs]
        descs = [pkg.make_desc(hs[0], hs[1:], job.Kinv, job.A, job.b, job.dmin, job.dmax,
                               radius=2, stride=1, iterations=0, seed=k) for k in (5, 6)]
        for counts in ((1, 2), (2, 1), (3, 3), (0, 0), (3, 0), (0, 3), (1, 2)):
            for d, n in zip(descs, counts):
                d.iterations = n
            outs = c.batch_run(descs, [job.shape] * 2, persistent=True)
            for d, o in zip(descs, outs):
                one = c.run_view(d, job.shape)
                for k in ("depth", "normal", "cost"):
                    assert np.array_equal(o[k], one[k]), (counts, k)
