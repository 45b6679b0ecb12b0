"""Ensembles: several runs of different grids in one context, stepped
concurrently through a HIP graph.  Every run must follow exactly the
trajectory it follows alone (bit for bit), across several graph replays
with downloads (synchronisations) between them, and with the graph off."""
import numpy as np
import pytest

from tests.configs import (HERNQUIST_SMALL, PLDF_SMALL, UDF_2SPECIES_DELAYED, UDF_C1, UDF_NOLINK,
                           UDF_ODD, UDF_TINY)

pytestmark = pytest.mark.gpu

V = pytest.importorskip("vlasolve_amd")

CFGS = [
    UDF_TINY,
    UDF_ODD,
    dict(HERNQUIST_SMALL, **{"grid.Pres": 32, "grid.Ures": [32, 16]}),
    dict(PLDF_SMALL, **{"grid.Pres": 24, "grid.Ures": [40, 6]}),
]


def alone(cfg, n):
    s = V.Solver(cfg)
    s.step(n)
    return s.f()


@pytest.mark.parametrize("graph", [True, False])
def test_ensemble_runs_match_single_runs(graph):
    print(f"case ensemble of {len(CFGS)} graph={graph}", flush=True)
    e = V.Ensemble(CFGS)
    e.set_graph(graph)
    done = 0
    for k in (3, 4, 1):  # replays separated by downloads
        e.step(k)
        done += k
        for i, cfg in enumerate(CFGS):
            fe = e.f(i)
            fa = alone(cfg, done)
            bad = np.count_nonzero(fe != fa)
            assert bad == 0, f"run {i} after {done} steps: {bad} points differ"


def test_calls_of_one_and_more_steps():
    """The captured first and last steps of a call, with and without linking
    and species, beside runs whose steps are all alike (one too wide for the
    slice step): calls of one step, two and several."""
    cfgs = [UDF_NOLINK, UDF_2SPECIES_DELAYED, UDF_C1,
            dict(UDF_C1, **{"grid.Pres": 150, "grid.Ures": [131, 3]})]
    print(f"case ensemble of {len(cfgs)}, calls of 1, 1, 2 and 4 steps", flush=True)
    e = V.Ensemble(cfgs)
    ones = [V.Solver(cfg) for cfg in cfgs]
    ctx = e.context
    for k in (1, 1, 2, 4, 1):
        e.step(k)
        for i, s in enumerate(ones):
            s.step(k)
            f = ctx.download_f(i, s.shape)
            assert np.array_equal(f, s.f()), (i, k)
            assert all(np.array_equal(a, b) for a, b in zip(ctx.get_chains(i), s.context.get_chains()))
