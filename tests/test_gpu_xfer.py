"""Copies of pageable memory through the page-locked ring: every byte arrives,
for sizes around its slots and chunks and past a whole turn of the ring, odd
addresses, page-locked memory, and several contexts copying at once."""
import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KIB, MIB = 1 << 10, 1 << 20
SIZES = [1, 3, 128 * KIB - 1, 128 * KIB, 128 * KIB + 1, MIB - 1, MIB, MIB + 1, 12 * MIB - 5,
         16 * MIB, 16 * MIB + 1, 37 * MIB + 3]


def round_trip(pkg, ctx, n, rng, offset=0):
    src = np.empty(n + offset, np.uint8)[offset:]
    src[:] = rng.integers(0, 256, n, dtype=np.uint8)
    dst = np.zeros(n + 2 * offset + 2, np.uint8)
    p = ctx.device_alloc(n)
    copy = pkg.lib().hp3d_pm_device_copy
    assert copy(ctx.h, ctypes.c_void_p(p), src.ctypes.data, n, 0) == 0
    assert copy(ctx.h, dst.ctypes.data + offset + 1, ctypes.c_void_p(p), n, 1) == 0
    ctx.device_free(p)
    assert np.array_equal(dst[offset + 1:offset + 1 + n], src)
    assert not dst[:offset + 1].any() and not dst[offset + 1 + n:].any()   # and nothing beside


@pytest.mark.parametrize("n", SIZES)
def test_round_trip(pkg, ctx, n):
    rng = np.random.default_rng(n)
    for offset in (0, 1, 61):
        round_trip(pkg, ctx, n, rng, offset)


def test_page_locked_memory(pkg, ctx):
    a, b = ctx.host_array((3 * MIB + 7,), np.uint8), ctx.host_array((3 * MIB + 7,), np.uint8)
    a[:] = np.random.default_rng(1).integers(0, 256, a.size, dtype=np.uint8)
    b[:] = 0
    p = ctx.device_alloc(a.size)
    ctx.upload_bytes(p, a)
    assert pkg.lib().hp3d_pm_device_copy(ctx.h, b.ctypes.data, ctypes.c_void_p(p), b.size, 1) == 0
    assert np.array_equal(a, b)
    ctx.device_free(p)
    ctx.host_free(a)
    ctx.host_free(b)


def test_contexts_copy_at_once(pkg):
    failed = []

    def one(seed):
        try:
            rng = np.random.default_rng(seed)
            with pkg.Context() as c:
                for _ in range(6):
                    round_trip(pkg, c, int(rng.integers(1, 24 * MIB)), rng)
        except BaseException as e:   # noqa: B902
            failed.append(repr(e))

    threads = [threading.Thread(target=one, args=(s,)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed


def test_overlapping_destinations_keep_the_later_output(pkg, ctx, scenes):
    """Two views of a batch given one array: it holds the second view's map."""
    job = scenes.plane_job(W=200, H=150, iterations=1)
    hs = [ctx.upload(im) for im in [job.ref] + job.srcs]
    descs = [pkg.make_desc(hs[0], hs[1:], job.Kinv, job.A, job.b, job.dmin, job.dmax, iterations=1,
                           seed=s) for s in (1, 2)]
    want = ctx.run_view(descs[1], job.shape)["depth"]
    got = np.zeros(job.shape, np.float32)
    outs = (pkg.ViewOut * 2)(*[pkg.ViewOut(pkg._p(got, pkg._f32p), None, None, None, 0)] * 2)
    rc = pkg.lib().hp3d_pm_batch_run(ctx.h, (pkg.ViewDesc * 2)(*descs), 2, outs, None)
    assert rc == 0
    assert np.array_equal(got, want)
    for h in hs:
        ctx.release(h)
