"""The solves and the kick by line tiles in LDS (grids whose slices fit neither
in a CU's LDS nor in the register kernels) at the sizes where they can go
wrong, bit for bit against the oracle: lines shorter than the pivots' head,
around the rows held in registers and past them, the fewest lines a tile may
have, short last tiles, one and two species.  No tolerance: the operations and
their order are the oracle's."""
import numpy as np
import pytest

from tests.configs import UDF_2SPECIES_DELAYED, UDF_C1, UDF_STRONG_KICK

pytestmark = pytest.mark.gpu

V = pytest.importorskip("vlasolve_amd")
from oracle import oracle as O  # noqa: E402

# cells of r, v and j (r and v lines have one node more)
GRIDS = [(3, 3, 2), (14, 15, 4), (15, 16, 9), (22, 24, 6), (30, 31, 5), (63, 40, 7), (94, 95, 3),
         (102, 103, 3), (110, 112, 2), (150, 131, 2), (131, 257, 2), (257, 130, 2), (340, 60, 2),
         (20, 619, 2), (619, 20, 2), (640, 20, 2)]
CASES = {"linking": UDF_C1, "no linking": UDF_C1, "strong kick": UDF_STRONG_KICK,
         "two species": UDF_2SPECIES_DELAYED}


@pytest.mark.parametrize("pr,pu,pj", GRIDS)
@pytest.mark.parametrize("case", list(CASES))
def test_line_tiles_bit_exact(monkeypatch, pr, pu, pj, case):
    monkeypatch.setenv("VLS_NO_SLICE_STEP", "1")
    cfg = dict(CASES[case], **{"grid.Pres": pr, "grid.Ures": [pu, pj],
                               "solver.noLinking": int(case == "no linking")})
    label = f"line tiles {pr + 1} x {pu + 1} x {pj} {case}"
    print("case " + label, flush=True)
    gpu, orc = V.Solver(cfg), O.Oracle(cfg, nthreads=0)
    for k in (1, 2):
        gpu.step(k)
        orc.step(k)
        assert np.array_equal(gpu.f(), orc.f()), label
    for a, b in zip(gpu.moments(), orc.last_moments()):
        assert np.array_equal(a, b), label


@pytest.mark.parametrize("pr,pu,pj", [(3, 3, 3), (14, 15, 4), (15, 17, 5), (24, 23, 6), (31, 25, 5),
                                      (40, 34, 9), (150, 131, 3), (64, 64, 4)])
def test_line_tiles_recorded(monkeypatch, pr, pu, pj):
    """The coefficients, a recorded run's state and its gradient against the
    streaming kernels, at the edges of the adjoint's chunks too (the gradient's sums in LDS have no fixed order: 1e-12
    of its largest, 5 steps of sums of some tens of terms)."""
    cfg = dict(UDF_C1, **{"grid.Pres": pr, "grid.Ures": [pu, pj]})
    print(f"case line tiles recorded {pr + 1} x {pu + 1} x {pj}", flush=True)
    monkeypatch.setenv("VLS_NO_SLICE_STEP", "1")
    seen, grads = [], []
    for stream in (None, "1"):
        if stream:
            monkeypatch.setenv("VLS_SPLINE_STREAM", stream)
        s = V.Solver(cfg)
        ctx = s.context
        s.step(4)
        got = [s.f(), ctx.coef(0, 2, s.nU, s.nR), *ctx.get_chains()]
        ctx.record(5, 2)
        got += [s.f(), *ctx.get_chains()]
        grads.append(ctx.adjoint(dL_df=np.cos(np.arange(s.f().size)))[0])
        seen.append(got)
    for k, (a, b) in enumerate(zip(*seen)):
        assert np.array_equal(a, b), k
    assert np.abs(grads[0] - grads[1]).max() <= 1e-12 * np.abs(grads[1]).max()


@pytest.mark.parametrize("pj", [1, 3])
def test_row_adjoints_of_register_shapes(monkeypatch, pj):
    """The rows of a register shape by tiles in LDS: the gradient has the bits
    of the register kernels (VLS_TILE_R leaves the tiles out)."""
    cfg = dict(UDF_C1, **{"grid.Pres": 128, "grid.Ures": [128, pj]})
    print(f"case row adjoints of a register shape, 129 x 129 x {pj}", flush=True)
    grads = []
    for tile in (None, "63"):
        if tile:
            monkeypatch.setenv("VLS_TILE_R", tile)
        s = V.Solver(cfg)
        s.context.record(4, 2)
        grads.append(s.context.adjoint(dL_df=np.cos(np.arange(s.f().size))))
    for a, b in zip(*grads):
        assert np.array_equal(a, b), np.abs(a - b).max()
