"""States and fields between host arrays and the device (nuc_upload_state,
nuc_download_state, nuc_average_field): bytes unchanged at the sizes where the
staged copies begin (16 MiB up, 8 MiB down), with last chunks of 8 and 16
bytes' alignment, into pinned memory, and from several threads at once."""
import ctypes
import threading

import numpy as np
import pytest

import nuc3d_amd as G

pytestmark = pytest.mark.gpu

# (staged once copies have lost time without it, as in test_gpu_staged.py: here the
# runtime copies)
SIZES = [(58, 58, 58),      # 7.8 MB: below both limits
         (61, 61, 59),      # 8.8 MB: above the limit down
         (75, 75, 75),      # 16.9 MB: above both, an odd number of values
         (128, 64, 64),     # 21 MB: exactly five chunks
         (103, 97, 101)]    # 40 MB: more chunks than workers, odd


def _values(n, seed):
    return np.random.default_rng(seed).random(5 * n[0] * n[1] * n[2]) + 1.0


@pytest.mark.parametrize("n", SIZES, ids=str)
@pytest.mark.parametrize("precision", [G.FP64, G.FP32], ids=["fp64", "fp32"])
def test_round_trip(n, precision):
    q = _values(n, 1)
    with G.Context(G.make_config(n=n, precision=precision)) as ctx:
        ctx.upload(q)
        want = q if precision == G.FP64 else q.astype(np.float32).astype(np.float64)
        assert np.array_equal(ctx.download(), want)


def test_pinned_array():
    G.lib()
    hip = ctypes.CDLL("libamdhip64.so.7")
    hip.hipHostMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t, ctypes.c_uint]
    hip.hipHostFree.argtypes = [ctypes.c_void_p]
    n, size = (75, 75, 75), 5 * 75 ** 3
    p = ctypes.c_void_p()
    assert hip.hipHostMalloc(ctypes.byref(p), 8 * size, 0) == 0
    pinned = np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_double)), (size,))
    q = _values(n, 2)
    with G.Context(G.make_config(n=n)) as ctx:
        pinned[:] = q
        ctx.upload(pinned)
        pinned[:] = 0.0
        G._check(G.lib().nuc_download_state(ctx.h, G._ptr(pinned)), "nuc_download_state", ctx.h)
        assert np.array_equal(pinned, q)
    assert hip.hipHostFree(p) == 0


def test_threads():
    n = (103, 97, 101)
    wrong = []

    def one(seed):
        q = _values(n, seed)
        with G.Context(G.make_config(n=n)) as ctx:
            for _ in range(3):
                ctx.upload(q)
                if not np.array_equal(ctx.download(), q):
                    wrong.append(seed)

    th = [threading.Thread(target=one, args=(s,)) for s in range(3)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not wrong


def test_odd_field_offset():
    """A field that starts 8 bytes off a 16-byte boundary."""
    n = (103, 103, 101)
    N = n[0] * n[1] * n[2]
    with G.Context(G.make_config(n=n)) as ctx:
        fields = np.random.default_rng(3).random(31 * N)
        ctx.average_restore(1, 1, fields)
        for i in (0, 1, 9):
            assert np.array_equal(ctx.average_field(0, i), fields[i * N:(i + 1) * N])
