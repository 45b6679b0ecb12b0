"""The streaming solves and kick (lines too long for a tile in LDS or
registers) at the sizes where they can go wrong, bit for bit against the
oracle: lines around the edges of a segment (16 rows of a column, 32 of a
row), shorter than the pivots' head, tiles of 64 lines that are partly empty,
have an odd last row or reach over several slices, and kicks of tens of cells
both ways.  No tolerance: the operations and their order are the oracle's."""
import numpy as np
import pytest

from tests.configs import UDF_C1, UDF_STRONG_KICK

pytestmark = pytest.mark.gpu

V = pytest.importorskip("vlasolve_amd")
from oracle import oracle as O  # noqa: E402

# cells of r, v and j (r and v lines have one node more)
GRIDS = [(3, 3, 2), (3, 62, 40), (14, 15, 4), (15, 16, 9), (30, 31, 5), (31, 32, 6), (32, 46, 5),
         (33, 47, 3), (40, 48, 3), (61, 63, 4), (63, 64, 3), (64, 65, 2), (95, 96, 3),
         (96, 128, 2), (130, 145, 3)]


@pytest.mark.parametrize("pr,pu,pj", GRIDS)
@pytest.mark.parametrize("case", ["linking", "no linking", "strong kick"])
def test_streams_bit_exact(monkeypatch, pr, pu, pj, case):
    monkeypatch.setenv("VLS_NO_SLICE_STEP", "1")
    monkeypatch.setenv("VLS_NO_REGISTER_LINES", "1")
    monkeypatch.setenv("VLS_SPLINE_STREAM", "1")
    base = UDF_STRONG_KICK if case == "strong kick" else UDF_C1
    cfg = dict(base, **{"grid.Pres": pr, "grid.Ures": [pu, pj],
                        "solver.noLinking": int(case == "no linking")})
    label = f"streams {pr + 1} x {pu + 1} x {pj} {case}"
    print("case " + label, flush=True)
    gpu, orc = V.Solver(cfg), O.Oracle(cfg, nthreads=0)
    for k in (1, 3):
        gpu.step(k)
        orc.step(k)
        assert np.array_equal(gpu.f(), orc.f()), label
    for a, b in zip(gpu.moments(), orc.last_moments()):
        assert np.array_equal(a, b), label


def test_streams_against_kernels_per_phase(monkeypatch):
    """The coefficients and the rings after a call, points of delay lines that
    were cleared (they keep the kicked value), a recorded run's state and its
    gradient: the same bits as the tiled solves and the kick in place; the
    gradient, whose sums in LDS have no fixed order, to 1e-12 of its largest
    (5 steps of sums of some tens of terms, each 1.1e-16 of its size off)."""
    cfg = dict(UDF_C1, **{"grid.Pres": 40, "grid.Ures": [34, 9]})
    print("case streams against kernels per phase", flush=True)
    monkeypatch.setenv("VLS_NO_SLICE_STEP", "1")
    monkeypatch.setenv("VLS_NO_REGISTER_LINES", "1")
    seen, grads = [], []
    for stream in ("1", "0"):
        monkeypatch.setenv("VLS_SPLINE_STREAM", stream)
        s = V.Solver(cfg)
        ctx = s.context
        s.step(4)
        got = [s.f(), ctx.coef(0, 3, s.nU, s.nR), *ctx.get_chains()]
        ctx.record(5, 2)
        got += [s.f(), *ctx.get_chains()]
        grads.append(ctx.adjoint(dL_df=np.cos(np.arange(s.f().size)))[0])
        ctx.clear_chains()
        s.step(3)
        got.append(s.f())
        seen.append(got)
    for k, (a, b) in enumerate(zip(*seen)):
        assert np.array_equal(a, b), k
    assert np.abs(grads[0] - grads[1]).max() <= 1e-12 * np.abs(grads[1]).max()
