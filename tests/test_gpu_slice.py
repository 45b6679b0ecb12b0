"""The step in two launches (k_kick_tile, k_slice_drift) at the sizes where it
can go wrong, bit for bit against the oracle: lines shorter than the pivots'
head, the edges of its chunks and of the rows held in registers, odd and even
pitches, several blocks per slice and more slices than CUs, with and without
linking, one and two species.  No tolerance: every schedule runs the same
operations in the same order."""
import numpy as np
import pytest

from tests.configs import UDF_2SPECIES_DELAYED, UDF_C1

pytestmark = pytest.mark.gpu

V = pytest.importorskip("vlasolve_amd")
from oracle import oracle as O  # noqa: E402

# cells of r, v and j (r and v lines have one node more)
GRIDS = [(3, 3, 2), (14, 15, 4), (15, 16, 5), (22, 23, 3), (23, 24, 6), (30, 31, 5), (63, 40, 7),
         (64, 33, 20), (95, 96, 3), (96, 97, 21), (103, 111, 2), (111, 112, 4), (180, 48, 9),
         (12, 13, 300)]


@pytest.mark.parametrize("pr,pu,pj", GRIDS)
@pytest.mark.parametrize("nolink", [0, 1])
def test_slice_step_bit_exact(pr, pu, pj, nolink):
    cfg = dict(UDF_C1, **{"grid.Pres": pr, "grid.Ures": [pu, pj], "solver.noLinking": nolink})
    _run(cfg, f"slice step {pr + 1} x {pu + 1} x {pj} noLinking {nolink}")


@pytest.mark.parametrize("pr,pu,pj", [(20, 17, 6), (96, 96, 5)])
def test_slice_step_two_species_bit_exact(pr, pu, pj):
    cfg = dict(UDF_2SPECIES_DELAYED, **{"grid.Pres": pr, "grid.Ures": [pu, pj]})
    _run(cfg, f"slice step, two species {pr + 1} x {pu + 1} x {pj}")


def _run(cfg, label):
    print("case " + label, flush=True)
    gpu, orc = V.Solver(cfg), O.Oracle(cfg, nthreads=0)
    for k in (1, 3):  # one step a call (its last), then several
        gpu.step(k)
        orc.step(k)
        assert np.array_equal(gpu.f(), orc.f()), label
    for a, b in zip(gpu.moments(), orc.last_moments()):
        assert np.array_equal(a, b), label
    # the statistics' sums (their groups of 16 rows and radii) at the same edges;
    # the entropy goes through the device's logarithm
    sg, so = gpu.stats_total(), orc.stats_total()
    for key in ("M", "E", "Ek", "Ep", "L1", "L2"):
        assert sg[key] == so[key], (label, key)
    assert abs(sg["S"] - so["S"]) <= 1e-14 * abs(so["S"])


def test_slice_step_against_kernels_per_phase(monkeypatch):
    """The coefficients and the rings after a call, points of delay lines that
    were cleared (they keep the kicked value) and a recorded run's state: the
    same bits as the kernels per phase."""
    cfg = dict(UDF_C1, **{"grid.Pres": 40, "grid.Ures": [34, 9]})
    print("case slice step against kernels per phase", flush=True)
    seen = []
    for off in (False, True):
        if off:
            monkeypatch.setenv("VLS_NO_SLICE_STEP", "1")
        s = V.Solver(cfg)
        ctx = s.context
        s.step(4)
        got = [s.f(), ctx.coef(0, 3, s.nU, s.nR), *ctx.get_chains()]
        ctx.record(5, 2)
        got += [s.f(), *ctx.get_chains()]
        ctx.clear_chains()
        s.step(3)
        got.append(s.f())
        seen.append(got)
    for k, (a, b) in enumerate(zip(*seen)):
        assert np.array_equal(a, b), k


@pytest.mark.parametrize("grid,by_slice", [
    ((64, 64, 256), True), ((64, 64, 257), False), ((32, 32, 1024), False),
    ((128, 32, 170), True), ((128, 32, 171), False), ((40, 35, 512), True), ((40, 35, 513), False),
    ((32, 48, 512), True), ((48, 32, 256), True), ((48, 32, 257), False),
    ((139, 32, 213), True), ((139, 32, 214), False), ((299, 24, 102), True), ((299, 24, 103), False)])
def test_slice_step_is_for_slices_that_fill_the_chip_once(grid, by_slice):
    """The grids that go by slice, at both sides of the bounds on the slices
    and on the kick's blocks (register lines and others)."""
    pr, pu, pj = grid
    print(f"case schedule of {pr + 1} x {pu + 1} x {pj}", flush=True)
    s = V.Solver(dict(UDF_C1, **{"grid.Pres": pr, "grid.Ures": [pu, pj]}))
    ctx = s.context
    ctx.set_timing(True)
    ctx.step(1)
    names = {n for n, _ in ctx.kernel_times()}
    assert ("slice_kick" in names) == by_slice, names


@pytest.mark.parametrize("pr,pu,pj", [(12, 13, 300), (16, 16, 600)])
def test_more_slices_than_cus_bit_exact(monkeypatch, pr, pu, pj):
    monkeypatch.setenv("VLS_SLICE_STEP", "1")
    _run(dict(UDF_C1, **{"grid.Pres": pr, "grid.Ures": [pu, pj]}),
         f"slice step {pr + 1} x {pu + 1} x {pj}")
