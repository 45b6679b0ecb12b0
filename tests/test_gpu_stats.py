"""The statistics of grids with more radii than the last kernel's LDS holds,
and at the bound: the oracle's sums bit for bit (the entropy goes through the
device's logarithm)."""
import pytest

from tests.configs import UDF_C1

pytestmark = pytest.mark.gpu

V = pytest.importorskip("vlasolve_amd")
from oracle import oracle as O  # noqa: E402


@pytest.mark.parametrize("pr,pj", [(15999, 680), (16000, 3), (23999, 4)])
def test_many_radii(pr, pj):
    cfg = dict(UDF_C1, **{"grid.Pres": pr, "grid.Ures": [4, pj]})
    print(f"case statistics of {pr + 1} x 5 x {pj}", flush=True)
    sg, so = V.Solver(cfg).stats_total(), O.Oracle(cfg, nthreads=0).stats_total()
    for key in ("M", "E", "Ek", "Ep", "L1", "L2"):
        assert sg[key] == so[key], key
    assert abs(sg["S"] - so["S"]) <= 1e-14 * abs(so["S"])
