"""Large transfers, downloads to pageable memory through the pinned pieces: f
comes back as it was sent at sizes around the smallest staged one, around whole pieces and shares of the
threads, and from two threads at once on contexts of their own (one of which
then takes the runtime's path)."""
import ctypes as C
import threading
import time

import numpy as np
import pytest

from tests.configs import UDF_C1

pytestmark = pytest.mark.gpu

V = pytest.importorskip("vlasolve_amd")


def _solver(pr, pu, pj):
    return V.Solver(dict(UDF_C1, **{"grid.Pres": pr, "grid.Ures": [pu, pj]}))


def _there_and_back(s, seed):
    f = np.random.default_rng(seed).standard_normal(s.shape)
    s.context.upload_f(0, f)
    assert np.array_equal(s.f(), f)


# 2 MiB - 32 KiB, 2 MiB, 2 MiB + 32 KiB, 3 MiB + 8 KiB, 16.6 MiB
@pytest.mark.parametrize("pr,pu,pj", [(63, 63, 63), (63, 63, 64), (63, 63, 65), (128, 63, 48),
                                      (128, 128, 131)])
def test_round_trip(pr, pu, pj):
    print(f"case transfer {pr + 1} x {pu + 1} x {pj}", flush=True)
    s = _solver(pr, pu, pj)
    for seed in range(2):
        _there_and_back(s, seed)


def test_two_threads():
    print("case transfer from two threads", flush=True)
    runs, wrong = [_solver(128, 128, 64), _solver(128, 96, 80)], []

    def work(k):
        try:
            for seed in range(5):
                _there_and_back(runs[k], 10 * k + seed)
        except AssertionError:
            wrong.append(k)

    th = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not wrong


def test_page_locked_memory_and_uploads_go_in_one_copy():
    """Page-locked arrays both ways, and uploads from pageable ones: as fast as
    the runtime's own copy of as many bytes (through pieces they took 1.8 to
    2.2 times as long), and whole."""
    L = V.lib()
    s = _solver(128, 128, 64)  # 8.1 MiB
    f = s.f()  # (the pinned pieces are there from here on)
    dev, locked = C.c_void_p(), C.c_void_p()
    assert L.hipMalloc(C.byref(dev), C.c_size_t(f.nbytes)) == 0
    assert L.hipHostMalloc(C.byref(locked), C.c_size_t(f.nbytes), C.c_uint(0)) == 0
    try:
        for pinned in (True, False):
            host = np.empty(s.shape)
            if pinned:
                buf = (C.c_double * f.size).from_address(locked.value)
                host = np.frombuffer(buf, np.float64).reshape(s.shape)
            f = np.random.default_rng(pinned).standard_normal(s.shape)
            host[:] = f
            at = C.c_void_p(host.ctypes.data)
            p = host.ctypes.data_as(C.POINTER(C.c_double))
            n = C.c_size_t(f.nbytes)
            pairs = [("upload", lambda: L.vls_upload_f(s.context._h, 0, p),
                      lambda: L.hipMemcpy(dev, at, n, C.c_int(1)))]
            if pinned:
                pairs.append(("download", lambda: L.vls_download_f(s.context._h, 0, p),
                              lambda: L.hipMemcpy(at, dev, n, C.c_int(2))))
                assert L.hipMemcpy(dev, at, n, C.c_int(1)) == 0
            for name, ours, runtime in pairs:
                best = [1e9, 1e9]
                for _ in range(20):
                    for k, fn in enumerate((ours, runtime)):
                        t = time.perf_counter()
                        assert fn() == 0
                        best[k] = min(best[k], time.perf_counter() - t)
                print(f"case {'page-locked' if pinned else 'pageable'} {name}: "
                      f"{best[0] * 1e3:.3f} ms, the runtime's copy {best[1] * 1e3:.3f}", flush=True)
                assert best[0] < 1.5 * best[1] + 3e-5
            host[:] = 0.0
            assert L.vls_download_f(s.context._h, 0, p) == 0
            assert np.array_equal(host, f)
    finally:
        L.hipFree(dev)
        L.hipHostFree(locked)
