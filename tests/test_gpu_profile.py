"""The profile call's two launches (k_slice_moment, k_moment_reduce) at the
edges of their tiles, and the launches of grids whose chunk sums don't fit in
one block's LDS: density, potential and enclosed mass from the oracle's moment
in the device order, bit for bit (the same operations in the same order)."""
import numpy as np
import pytest

from tests.configs import UDF_C1

pytestmark = pytest.mark.gpu

V = pytest.importorskip("vlasolve_amd")
torch = pytest.importorskip("torch")
from oracle import oracle as O  # noqa: E402


@pytest.mark.parametrize("pr,pu,pj", [(3, 3, 1), (15, 16, 19), (16, 17, 20), (62, 15, 21),
                                      (63, 31, 41), (125, 8, 40), (599, 8, 300)])
def test_profile_matches_oracle(pr, pu, pj):
    print(f"case profile {pr + 1} x {pu + 1} x {pj}", flush=True)
    cfg = dict(UDF_C1, **{"grid.Pres": pr, "grid.Ures": [pu, pj]})
    s, orc = V.Solver(cfg), O.Oracle(cfg, nthreads=0)
    dM, M, _ = orc.moments()
    rho, phi = O.density_potential(orc.axes()[0], dM, M)
    f = torch.from_numpy(s.f()).to("cuda")
    out = torch.full((3, s.nR), float("nan"), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    for _ in range(2):
        s.context.density_potential_noalloc(f.data_ptr(), *(x.data_ptr() for x in out))
    s.context.synchronize()
    got = out.cpu().numpy()
    assert np.array_equal(got[2], M)
    assert np.array_equal(got[0], rho) and np.array_equal(got[1], phi)
