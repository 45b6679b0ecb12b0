"""The schedule tuner (vls_autotune): runs of shapes with and without
register line solvers, tuned, follow bit for bit the trajectories of the
same runs with the default schedules (every schedule runs the same
operations per line in the same order), inside the ensemble's graph; the
choices are cached per shape."""
import numpy as np
import pytest

from tests.configs import HERNQUIST_SMALL, UDF_2SPECIES_DELAYED, UDF_C1, UDF_ODD, UDF_TINY

pytestmark = pytest.mark.gpu

V = pytest.importorskip("vlasolve_amd")

CFGS = [UDF_TINY, UDF_ODD, dict(UDF_C1, **{"grid.Pres": 96, "grid.Ures": [128, 24]}),
        dict(HERNQUIST_SMALL, **{"grid.Pres": 64, "grid.Ures": [64, 32]})]


def test_tuned_schedules_give_the_same_bits():
    n = 12
    print(f"case autotune of {len(CFGS)} runs, {n} graph steps", flush=True)
    ref = V.Ensemble(CFGS)
    ref.step(n)
    e = V.Ensemble(CFGS)
    desc = e.autotune()
    print("  " + desc, flush=True)
    assert desc.count(";") == len(CFGS) - 1
    e.step(n)
    for k in range(len(CFGS)):
        assert np.array_equal(e.f(k), ref.f(k)), k
    # a second tuning of the same shapes comes from the cache
    again = V.Ensemble(CFGS[:1])
    assert "cached" in again.autotune()


@pytest.mark.parametrize("pr,pu,pj", [(24, 20, 12), (64, 64, 6), (150, 131, 3)])
def test_two_species(pr, pu, pj):
    """Runs of two species, whose moment reads both planes of f: by slice,
    register lines, and lines too long for either."""
    cfg = dict(UDF_2SPECIES_DELAYED, **{"grid.Pres": pr, "grid.Ures": [pu, pj]})
    print(f"case autotune of two species, {pr + 1} x {pu + 1} x {pj}", flush=True)
    ref, s = V.Solver(cfg), V.Solver(cfg)
    print("  " + s.context.autotune(), flush=True)
    ref.step(3)
    s.step(3)
    assert np.array_equal(s.f(), ref.f())
    assert all(np.array_equal(a, b) for a, b in zip(s.context.get_chains(), ref.context.get_chains()))


def test_choices_are_kept_apart():
    """A choice made for two species, without linking or for a run that has the
    GPU for itself is not taken for the same grid under other conditions."""
    grid = {"grid.Pres": 28, "grid.Ures": [26, 10]}
    runs = [dict(UDF_2SPECIES_DELAYED, **grid), dict(UDF_C1, **grid),
            dict(UDF_C1, **grid, **{"solver.noLinking": 1})]
    print("case autotune of one grid under several conditions", flush=True)
    for again in (False, True):
        for cfg in runs:
            desc = V.Solver(cfg).context.autotune()
            print("  " + desc, flush=True)
            assert ("cached" in desc) == again and " 0.0 us" not in desc
    # runs that share the GPU go by slice where the sizes say so, whatever one
    # of them alone was timed at
    desc = V.Ensemble(runs[1:2] * 3).autotune()
    print("  " + desc, flush=True)
    assert desc.count("slice step (by its sizes") == 3
