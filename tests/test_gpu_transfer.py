"""Large transfers through the pinned pieces: f comes back as it was sent at
sizes around the smallest staged one, around whole pieces and shares of the
threads, and from two threads at once on contexts of their own (one of which
then takes the runtime's path)."""
import threading

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
