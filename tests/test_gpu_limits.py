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
