"""The C-ABI library on the CPU: it loads, exports every function the public
header declares, and its host-side helpers behave; device calls fail cleanly
where there is no GPU."""
import ctypes as C
import re
from pathlib import Path

import numpy as np
import pytest

import vlasolve_amd as V

HEADER = Path(__file__).resolve().parents[1] / "include" / "vlasolve_hip.h"


def declared_functions():
    text = HEADER.read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(vlsd?_\w+)\s*\(", text)))


def test_exports_every_declared_function():
    lib = V.lib()
    names = declared_functions()
    assert len(names) >= 30
    missing = [n for n in names if not hasattr(lib, n)]
    assert not missing, missing
    assert set(names) <= set(V.EXPORTS) | set(names)


def test_no_device_is_reported():
    if V.lib().vls_create and _has_gpu():
        pytest.skip("a GPU is present")
    with pytest.raises(V.VlsError, match="no HIP device"):
        V.Solver({"grid.Pres": 8, "grid.Ures": [8, 4]})


def _has_gpu():
    try:
        V.device_info()
        return True
    except V.VlsError:
        return False


def thomas(dim, hinv):
    L = V.lib()
    P = C.POINTER(C.c_double)
    L.vls_thomas_table.argtypes = [C.c_int, C.c_double, P, P, P, P]
    u, d, rd, cs = np.zeros(dim + 2), np.zeros(dim + 2), np.zeros(dim + 2), np.zeros(8)
    assert L.vls_thomas_table(dim, hinv, *(a.ctypes.data_as(P) for a in (u, d, rd, cs))) == 0
    return u, d, rd, cs


def test_pivot_table_fixed_point():
    # the pivots of the natural spline solve settle exactly after a few rows and
    # do not depend on the knot spacing
    u1, d1, rd1, c1 = thomas(201, 31.4)
    u2, d2, rd2, c2 = thomas(65, 3.0)
    assert d1[1] == 1.0 and u1[1] == 0.0  # first interior row after the natural row
    assert np.all(d1[17:202] == d1[201]) and np.all(u1[17:202] == u1[201])
    assert np.array_equal(d1[1:40], d2[1:40])
    assert np.all(rd1[1:202] == 1.0 / d1[1:202])


def test_known_divisor_division_is_correctly_rounded():
    L = V.lib()
    P = C.POINTER(C.c_double)
    L.vls_check_division.argtypes = [P, C.c_int, C.c_int64, C.c_uint64, C.POINTER(C.c_int64)]
    divs = []
    for dim, hinv in [(201, 25.0), (513, 60.0), (17, 2.0)]:
        u, d, rd, cs = thomas(dim, hinv)
        divs += list(d[1:dim + 1]) + [cs[6]]
    divs += list(np.random.default_rng(0).uniform(1e-3, 1e3, 200))
    b = np.array(divs)
    bad = C.c_int64(-1)
    assert L.vls_check_division(b.ctypes.data_as(P), len(b), 20000, 99, C.byref(bad)) == 0
    assert bad.value == 0


def test_ndfield_roundtrip(tmp_path):
    from vlasolve_amd import ndfield

    a = np.random.default_rng(1).uniform(size=(4, 5, 6))
    p = tmp_path / "x.ND"
    ndfield.write(p, a, [0.01, -2, 0], [24.99, 4, 1.6], comment="1 1 0 1 2 0")
    b, meta = ndfield.read(p)
    assert np.array_equal(a, b) and meta["dims"] == [6, 5, 4]
    assert meta["comment"] == "1 1 0 1 2 0"


def test_two_operation_pivot_division_is_correctly_rounded():
    """The line solves divide by a pivot d as fma(a, rh, RN(a rl)) with
    rh = RN(1/d), rl = RN(1/d - rh).  Exact rational arithmetic: the value
    before the fma's rounding is off by less than three of the smallest
    distances of a quotient from a midpoint, and the numerators at the first
    distance (the only ones that could round wrongly) round to a/d."""
    from fractions import Fraction as F

    pivots = sorted(set(thomas(201, 31.4)[1][1:202]) | set(thomas(5, 3.0)[1][1:6]))
    solved = 0  # pivots whose numerators at the first distance were sought
    for d in pivots:
        d = float(d)
        D = int(F(d) * F(2) ** (53 - int(np.frexp(d)[1])))
        t = (D & -D).bit_length() - 1
        rh = 1.0 / d
        rl = float((1 - F(rh) * F(d)) / F(d))  # float() rounds to nearest
        bound = 4 * abs(F(rl) * F(d)) * D
        assert bound < 3 * 2 ** t
        rng = np.random.default_rng(3)
        tests = [int(a) for a in rng.integers(2 ** 52, 2 ** 53, 200)]
        if bound >= 2 ** t:
            solved += 1
            odd = D >> t
            for k in (53, 54):
                inv = pow(2, -(k - t), odd)
                for a0 in (inv, odd - inv):
                    lo = a0 + -(-(2 ** 52 - a0) // odd) * odd
                    found = list(range(lo, 2 ** 53, odd))
                    assert len(found) <= 2 ** (t + 1)
                    tests += found
        for A in tests:
            a = float(A)
            assert float(F(a) * F(rh) + F(a * rl)) == a / d, (d, A)
    assert len(pivots) >= 16 and solved >= 2


def test_pivot_division_host_check():
    """The compiled division by a pivot and the condition that the set-up puts to
    every pivot: the pivots are proven and divide as IEEE over random numerators
    and those nearest to a rounding tie; a remainder that is not the rounded one
    is refused; so are divisors that do divide wrongly."""
    L = V.lib()
    P = C.POINTER
    L.vls_check_pivot_division.argtypes = [P(C.c_double), C.c_int, C.c_int, C.c_int64, C.c_uint64,
                                           P(C.c_int), P(C.c_int64)]

    def check(divisors, ulps=0, samples=20000):
        d = np.array(divisors, np.float64)
        proven, bad = np.full(len(d), -1, np.int32), np.full(len(d), -1, np.int64)
        assert L.vls_check_pivot_division(d.ctypes.data_as(P(C.c_double)), len(d), ulps, samples, 5,
                                          proven.ctypes.data_as(P(C.c_int)),
                                          bad.ctypes.data_as(P(C.c_int64))) == 0
        return proven, bad

    pivots = sorted({float(x) for x in thomas(513, 60.0)[1][1:514]})
    assert len(pivots) >= 16
    proven, bad = check(pivots)
    assert np.all(proven == 1) and np.all(bad == 0)
    for ulps in (-1, 1, 1000):
        assert not np.any(check(pivots, ulps, 0)[0])
    # divisors in [1, 2): none that is proven divides wrongly, and some that are
    # not proven do
    d = np.random.default_rng(1).uniform(1.0, 2.0, 20000)
    proven, bad = check(d, samples=20)
    assert np.all(bad[proven == 1] == 0)
    assert np.count_nonzero(bad) > 50 and 0.95 < proven.mean() < 1.0
    for odd in (0.0, 5e-324, np.inf, np.nan):
        assert L.vls_check_pivot_division((C.c_double * 1)(odd), 1, 0, 0, 1, (C.c_int * 1)(),
                                          (C.c_int64 * 1)()) == 1
