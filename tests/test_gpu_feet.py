"""Foot tables and delay lines changed between steps, and feet and back cells
at the edges of the domain that vls_set_drift and vls_set_chains accept: every
schedule, and the captured step of an ensemble, gives the bits of the kernels
per phase.  No tolerance: the schedules run the same operations."""
import ctypes as C

import numpy as np
import pytest

from tests.configs import UDF_C1

pytestmark = pytest.mark.gpu

V = pytest.importorskip("vlasolve_amd")

OUT, CHAIN = 1, 2
NO_LINES = {"VLS_NO_SLICE_STEP": "1", "VLS_NO_REGISTER_LINES": "1"}
PHASES = dict(NO_LINES, VLS_SPLINE_STREAM="0")
SCHEDULES = {"slice": {}, "streams": dict(NO_LINES, VLS_SPLINE_STREAM="1")}


def _cfg(pr=40, pu=34, pj=9):
    return dict(UDF_C1, **{"grid.Pres": pr, "grid.Ures": [pu, pj]})


def _p(a, t=C.c_double):
    return a.ctypes.data_as(C.POINTER(t))


def _feet(shape, seed, chains=()):
    """A foot table inside the domain, a tenth of it outside the grid, the
    given points on delay lines."""
    rng = np.random.default_rng(seed)
    nJ, nU, nR = shape
    n = nJ * nU * nR
    xr, xu = rng.uniform(0, nR - 1, n), rng.uniform(0, nU - 1, n)
    flag = np.where(rng.random(n) < 0.1, OUT, 0).astype(np.uint8)
    flag[list(chains)] = CHAIN
    return xr, xu, flag


def _set_drift(ctx, run, xr, xu, flag):
    V._check(V.lib().vls_set_drift(ctx._h, run, _p(xr), _p(xu), _p(flag, C.c_uint8)))


def _set_chains(ctx, run, points, shape, seed, back=None):
    rng = np.random.default_rng(seed)
    nJ, nU, nR = shape
    n = len(points)
    length = rng.integers(2, 6, n).astype(np.int32)
    head = (rng.integers(0, 6, n) % length).astype(np.int32)
    bxr, bxu = rng.uniform(0, nR - 1, n), rng.uniform(0, nU - 1, n)
    if back is not None:
        bxr[:], bxu[:] = back
    out = np.zeros(n, np.uint8)
    vals = rng.random(int(length.sum()))
    V._check(V.lib().vls_set_chains(ctx._h, run, n, _p(np.asarray(points, np.int64), C.c_int64),
                                    _p(length, C.c_int32), _p(head, C.c_int32), _p(bxr), _p(bxu),
                                    _p(out, C.c_uint8), _p(vals)))


def _points(shape, n, seed, taken=()):
    rng = np.random.default_rng(seed)
    free = np.setdiff1d(np.arange(int(np.prod(shape))), np.asarray(taken, np.int64))
    return np.sort(rng.choice(free, n, replace=False))


def _under(monkeypatch, env, fn):
    with monkeypatch.context() as m:
        for k, v in env.items():
            m.setenv(k, v)
        return fn()


def _same(a, b):
    for k, (x, y) in enumerate(zip(a, b)):
        assert np.array_equal(x, y), (k, np.flatnonzero(np.asarray(x) != np.asarray(y))[:5])


@pytest.mark.parametrize("schedule", list(SCHEDULES))
def test_captured_step_follows_new_feet(monkeypatch, schedule):
    """An ensemble whose foot table gets delay-line points without lines
    between two calls: the points keep their kicked value, as in the same
    steps without the captured graph."""
    cfgs = [_cfg(), _cfg(33, 30, 6)]
    print(f"case captured step, new feet, {schedule}", flush=True)

    def run(graph):
        e = V.Ensemble(cfgs)
        e.set_graph(graph)
        ctx = e.context
        shapes = [e.f(k).shape for k in range(2)]
        for k, shape in enumerate(shapes):
            ctx.clear_chains(k)
            _set_drift(ctx, k, *_feet(shape, k))
        e.step(2)
        for k, shape in enumerate(shapes):
            _set_drift(ctx, k, *_feet(shape, k, _points(shape, 400, 7 + k)))
        e.step(3)
        return [e.f(0), e.f(1)]

    want = _under(monkeypatch, PHASES, lambda: run(False))
    _same(_under(monkeypatch, SCHEDULES[schedule], lambda: run(True)), want)


@pytest.mark.parametrize("schedule", list(SCHEDULES))
def test_moved_delay_line_points(monkeypatch, schedule):
    """Lines attached to one set of points and a later foot table whose
    delay-line points are others, as many as there are lines or fewer: the
    points without a line keep their kicked value."""
    print(f"case moved delay-line points, {schedule}", flush=True)

    def run():
        s = V.Solver(_cfg())
        ctx, shape = s.context, s.shape
        ctx.clear_chains()
        lines = _points(shape, 60, 1)
        _set_drift(ctx, 0, *_feet(shape, 2, lines))
        _set_chains(ctx, 0, lines, shape, 3)
        s.step(2)
        _set_drift(ctx, 0, *_feet(shape, 4, _points(shape, 50, 5, lines)))
        s.step(3)
        return [s.f(), *ctx.get_chains()]

    want = _under(monkeypatch, PHASES, run)
    _same(_under(monkeypatch, SCHEDULES[schedule], run), want)


def test_back_cell_below_the_first_knot(monkeypatch):
    """A back cell inside (-1, 0): its integer part is 0, so it is evaluated."""
    print("case back cell below the first knot", flush=True)

    def run():
        s = V.Solver(_cfg())
        ctx, shape = s.context, s.shape
        lines = _points(shape, 40, 1)
        _set_drift(ctx, 0, *_feet(shape, 2, lines))
        ctx.clear_chains()
        _set_chains(ctx, 0, lines, shape, 3, back=(-0.375, 3.25))
        s.step(7)
        return [s.f(), *ctx.get_chains()]

    _same(_under(monkeypatch, {}, run), _under(monkeypatch, PHASES, run))


@pytest.mark.parametrize("axis", [0, 1])
@pytest.mark.parametrize("where", ["feet", "back cells"])
def test_past_the_last_knot(monkeypatch, axis, where):
    """Feet and back cells between the last knot and the next integer: their
    stencil ends in the first column of the next row, or the first row of the
    next slice."""
    print(f"case past the last knot, axis {axis}, {where}", flush=True)

    def run():
        s = V.Solver(_cfg(39, 34, 9))  # rows of 42 coefficients, an odd pitch in LDS
        ctx, shape = s.context, s.shape
        lines = _points(shape, 40, 1)
        feet = _feet(shape, 2, lines)
        last = (shape[2] - 1, shape[1] - 1)
        back = [5.5, 6.5]
        if where == "feet":
            feet[axis][::7] = last[axis] + 0.375
        else:
            back[axis] = last[axis] + 0.375
        ctx.clear_chains()
        _set_drift(ctx, 0, *feet)
        _set_chains(ctx, 0, lines, shape, 3, back=back)
        s.step(7)
        return [s.f(), *ctx.get_chains()]

    _same(_under(monkeypatch, {}, run), _under(monkeypatch, PHASES, run))
