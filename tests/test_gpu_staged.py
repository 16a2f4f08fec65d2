"""Copies that do go through the staging memory, which is pinned only once copies
have lost some time without it and given back with the last context: a context of
the module holds it, past that mark.  Bytes at the sizes where staging begins and chunks
end, a pinned array beside it, and contexts that come and go during a copy."""
import ctypes
import threading
import time

import numpy as np
import pytest

import nuc3d_amd as G
from test_gpu_transfer import SIZES, _values

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def staging():
    n = (128, 128, 128)   # 84 MB
    with G.Context(G.make_config(n=n)) as ctx:
        q = _values(n, 9)
        for _ in range(4):
            ctx.upload(q)
            assert np.array_equal(ctx.download(), q)
        yield


@pytest.mark.parametrize("n", SIZES + [(128, 128, 64)], ids=str)   # 42 MB: ten chunks
@pytest.mark.parametrize("precision", [G.FP64, G.FP32], ids=["fp64", "fp32"])
def test_round_trip(n, precision):
    with G.Context(G.make_config(n=n, precision=precision)) as ctx:
        for seed in (1, 2):   # the slots hold the first's bytes
            q = _values(n, seed)
            ctx.upload(q)
            want = q if precision == G.FP64 else q.astype(np.float32).astype(np.float64)
            assert np.array_equal(ctx.download(), want)


def test_odd_field_offset():
    """Averaged fields whose chunks begin 8 bytes off a 16-byte boundary."""
    n = (103, 103, 101)
    N = n[0] * n[1] * n[2]
    with G.Context(G.make_config(n=n)) as ctx:
        fields = np.random.default_rng(3).random(31 * N)
        ctx.average_restore(1, 1, fields)
        for i in (0, 1, 9):
            assert np.array_equal(ctx.average_field(0, i), fields[i * N:(i + 1) * N])


def _hip():
    """The HIP runtime that the library is linked to, as this process mapped it."""
    with open("/proc/self/maps") as f:
        return ctypes.CDLL(next(ln.split()[-1] for ln in f if "libamdhip64" in ln))


def test_pinned_array():
    hip = _hip()
    n, size = (75, 75, 75), 5 * 75 ** 3
    p = ctypes.c_void_p()
    assert hip.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(8 * size), 0) == 0
    pinned = np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_double)), (size,))
    q = _values(n, 2)
    with G.Context(G.make_config(n=n)) as ctx:
        pinned[:] = q
        ctx.upload(pinned)
        pinned[:] = 0.0
        G._check(G.lib().nuc_download_state(ctx.h, G._ptr(pinned)), "nuc_download_state", ctx.h)
        assert np.array_equal(pinned, q)
    assert hip.hipHostFree(p) == 0


def test_contexts_beside_a_waiting_download():
    """A download behind queued steps holds up neither a context's creation and
    destruction nor a serving loop's."""
    n = (192, 192, 192)
    cfg = G.make_config(n=n, scheme=G.CRWENO5, vis=G.CD6, model=G.NAVIERSTOKES3D, mach=0.2, reynolds=400.0)
    with G.Context(cfg) as ctx:
        ctx.upload(G.init_tgv(cfg))
        ctx.step(2)
        ctx.step_async(200)   # about a second
        done = threading.Event()

        def down():
            ctx.download()
            done.set()

        th = threading.Thread(target=down)
        th.start()
        time.sleep(0.1)   # into its copy
        t = time.perf_counter()
        G.Context(G.make_config(n=(16, 16, 16))).close()
        G.Server().close()
        t = time.perf_counter() - t
        before = not done.is_set()
        th.join()
        print(f"context and serving loop created and destroyed in {1e3 * t:.1f} ms", flush=True)
        assert before
