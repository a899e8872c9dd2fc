"""Copies through the pinned ring: accumulator texels written and read back bit for
bit at sizes around its edges (a copy the runtime makes, one chunk, two, more than
the ring holds and a ragged last one), into and out of unaligned host memory, and
from two contexts at once."""
import threading

import numpy as np
import pytest

import pathtracer_amd as pt

# texels: below the threshold, at it, one chunk less / more a texel, two chunks, the ring, ragged beyond
SIZES = [(1, 1), (64, 128), (8191, 1), (131072, 1), (131073, 1), (262147, 1), (1048577, 1), (1237, 1531)]


def round_trip(ctx, w, h, seed):
    rng = np.random.default_rng(seed)
    acc = ctx.accum(w, h)
    n = w * h * 4
    raw = rng.integers(0, 2 ** 32, n + 1, dtype=np.uint64).astype(np.uint32)
    src = raw.view(np.uint8)[1:1 + 4 * n].view()  # one byte off alignment
    ctx.check(pt.lib.pt_accum_write_xyz(acc.h, pt.C.cast(src.ctypes.data, pt.C.POINTER(pt.C.c_float)), n))
    out = np.zeros(4 * n + 3, np.uint8)
    ctx.check(pt.lib.pt_accum_read_xyz(acc.h, pt.C.cast(out.ctypes.data + 3, pt.C.POINTER(pt.C.c_float)), n))
    assert np.array_equal(out[3:], src)
    assert np.array_equal(acc.read().view(np.uint8).reshape(-1), src)
    acc.release()


@pytest.mark.gpu
@pytest.mark.parametrize("w,h", SIZES)
def test_round_trip(gpu_ctx, w, h):
    round_trip(gpu_ctx, w, h, w + h)


@pytest.mark.gpu
def test_two_contexts_in_two_threads():
    errors = []

    def work(seed):
        try:
            with pt.Context(0) as ctx:
                for i in range(6):
                    round_trip(ctx, 700 + 31 * i, 400 + seed, seed * 10 + i)
        except BaseException as e:  # noqa: BLE001
            errors.append(e)

    t = [threading.Thread(target=work, args=(s,)) for s in (1, 2)]
    [x.start() for x in t]
    [x.join() for x in t]
    assert not errors, errors


@pytest.mark.gpu
@pytest.mark.parametrize("w,h", [(64, 128), (1237, 1531)])
def test_page_locked_memory(gpu_ctx, w, h):
    """The same bytes into and out of page-locked memory, which the runtime copies itself."""
    n = w * h * 4
    p = pt.C.c_void_p()
    assert pt.lib.hipHostMalloc(pt.C.byref(p), pt.C.c_size_t(n * 4), 0) == 0  # of the runtime the library uses
    try:
        bits = np.random.default_rng(3).integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32)
        host = np.ctypeslib.as_array(pt.C.cast(p, pt.C.POINTER(pt.C.c_uint32)), (n,))
        host[:] = bits
        acc = gpu_ctx.accum(w, h)
        gpu_ctx.check(pt.lib.pt_accum_write_xyz(acc.h, pt.C.cast(p, pt.C.POINTER(pt.C.c_float)), n))
        host[:] = 0
        assert np.array_equal(acc.read().view(np.uint32).reshape(-1), bits)
        gpu_ctx.check(pt.lib.pt_accum_read_xyz(acc.h, pt.C.cast(p, pt.C.POINTER(pt.C.c_float)), n))
        assert np.array_equal(host, bits)
        acc.release()
    finally:
        pt.lib.hipHostFree(p)
