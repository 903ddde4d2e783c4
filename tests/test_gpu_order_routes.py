"""The order and maximum stages over their routes: programs that run on value
streams, on the record sweep and on the general kernels, row counts around the
selection's and the row kernels' block sizes, and rows with many ties, bit for
bit against the oracle for programs of + - * and / (the level's ends to the
rounding of their derivative)."""
import math

import numpy as np
import pytest

import oracle
from rcsr_hip import host
from rcsr_hip.expr import ADD, DIV, LOG, MUL, SQUARE, SUB, const, node, var

pytestmark = pytest.mark.gpu


def _deep(levels):
    """A right-deep tree: it keeps `levels` values below its top."""
    t = node(MUL, const(0.5), var(0))
    for i in range(levels):
        t = node(ADD if i % 2 else SUB, node(MUL, const(0.1 * (i + 1)), var(i % 2)), t)
    return t


TREES = {
    "line": node(ADD, node(MUL, const(1.5), var(0)), const(-0.25)),
    "ratio": node(DIV, node(MUL, const(0.7), var(1)),
                  node(ADD, const(2.0), node(MUL, var(0), var(0)))),
    "constant": node(MUL, const(0.0), var(0)),
    "stream limit": _deep(4),
    "stack limit": _deep(8),
    "general": _deep(11),
}


def _setup(n, ties):
    rng = np.random.default_rng(n)
    x = rng.standard_normal((2, n))
    y = rng.standard_normal(n)
    if ties:
        x, y = np.round(x), np.round(2.0 * y) / 2.0
    ev = host.GpuEvaluator(x.astype(np.float32).reshape(-1), n, 2, y.astype(np.float32))
    assert ev.set_fit_data(x.reshape(-1), y)
    return x.T.copy(), y, ev


@pytest.mark.parametrize("ties", [False, True])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 63, 257, 512, 513, 2049, 4096, 4097, 20011])
def test_medians_and_quartile_means_over_every_route(n, ties):
    x, y, ev = _setup(n, ties)
    plans = [host.gpu_fit_plan(t) for t in TREES.values()]
    print(f"order routes: {n} rows, ties {ties}", flush=True)
    for what, f in ((0, oracle.median_abs), (1, oracle.iqr_mean_abs)):
        val, st, ms = ev.order_stat_batch(plans, what)
        assert ms >= 0 and not st.any()
        for v, (name, t) in zip(val, TREES.items()):
            assert v == f(oracle.predict_flat(t, x) - y), (name, what)
    outs, ms = ev.max_scan_batch(plans)
    assert ms >= 0
    for o, (name, t) in zip(outs, TREES.items()):
        vm, row, lo, hi, stt = oracle.max_scan(oracle.predict_flat(t, x) - y)
        assert (o.vmax, o.row, o.status) == (vm, row, 0), name
        assert (o.lo, o.hi) == (-math.inf, math.inf)
    ev.close()


@pytest.mark.parametrize("ties", [False, True])
@pytest.mark.parametrize("n", [1, 130, 1025])
def test_level_intervals_over_every_route(n, ties):
    x, y, ev = _setup(n, ties)
    names = [k for k in TREES if k != "constant"]
    plans = [host.gpu_fit_plan(TREES[k]) for k in names]
    for scale in (0.9, 1.3):
        resid = [oracle.predict_flat(TREES[k], x) - y for k in names]
        levels = [scale * float(np.max(np.abs(r))) for r in resid]
        outs, ms = ev.max_scan_batch(plans, coords=[0] * len(names), levels=levels)
        assert ms >= 0
        for k, r, lv, o in zip(names, resid, levels, outs):
            b = np.array([oracle.gradients(TREES[k], x[i])[0][0] for i in range(n)])
            vm, row, lo, hi, stt = oracle.max_scan(r, b, lv)
            assert (o.vmax, o.row, o.status) == (vm, row, 0), k
            if math.isinf(lo):
                assert (o.lo, o.hi) == (lo, hi), k
            else:
                # a handful of roundings in b and in the quotient
                assert o.lo == pytest.approx(lo, rel=1e-14) and o.hi == pytest.approx(hi, rel=1e-14)
    ev.close()


def test_rows_that_are_not_finite_and_huge_derivatives():
    x, y, ev = _setup(700, False)
    trees = [node(MUL, const(1.0), node(LOG, var(0))), TREES["line"],
             # a derivative of 1e-320: its product leaves the normal range
             node(MUL, const(1e-290), node(MUL, node(SQUARE, const(1e-30)), var(0)))]
    plans = [host.gpu_fit_plan(t) for t in trees]
    val, st, ms = ev.order_stat_batch(plans, 0)
    assert list(st) == [2, 0, 0] and math.isnan(val[0]) and np.isfinite(val[1:]).all()
    outs, ms = ev.max_scan_batch(plans, coords=[0, 0, 1], levels=[1.0, 9.0, 9.0])
    assert [o.status for o in outs] == [2, 0, 0] and outs[0].row == -1
    assert math.isnan(outs[0].vmax) and math.isfinite(outs[1].vmax)
    b = np.array([oracle.gradients(trees[2], r)[0][1] for r in x])
    vm, row, lo, hi, stt = oracle.max_scan(oracle.predict_flat(trees[2], x) - y, b, 9.0)
    assert (outs[2].vmax, outs[2].row, outs[2].lo, outs[2].hi) == (vm, row, lo, hi)
    ev.close()
