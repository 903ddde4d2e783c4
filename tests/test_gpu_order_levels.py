"""Level intervals of the maximum scan where the constant's derivative has a
partial of zero, one that is not finite, or a product that leaves the range of
f64 on the way up or down the tree.  The record sweep takes the product of the
partials from the leaf up, the general kernel from the root down: a program
gives the same answer on both routes (with a deep zero term added it runs on
the general kernel), and the oracle's."""
import math

import numpy as np
import pytest

import oracle
from rcsr_hip import host
from rcsr_hip.expr import (ABS, ADD, COS, COSH, CUBE, DIV, ERF, ERFC, EXP, GAUSS, MUL, NEG, POW, SIG,
                           SIN, SINH, SQRT, SQUARE, SUB, TAN, TANH, const, node, var)

pytestmark = pytest.mark.gpu

ROWS = 200


def _line(c=1.2, x=None):
    return node(MUL, const(c), var(0) if x is None else x)


def _scaled(t, *factors):
    for f in factors:
        t = node(MUL, t, const(f))
    return t


def _on_the_general_kernel(t):
    """t + 0 * deep, where deep keeps eleven values below its top."""
    deep = var(1)
    for i in range(11):
        deep = node(ADD if i % 2 else SUB, node(MUL, const(0.1 * (i + 1)), var(i % 2)), deep)
    return node(ADD, t, node(MUL, const(0.0), deep))


def _rows():
    rng = np.random.default_rng(41)
    x = rng.standard_normal((ROWS, 2))
    x[:, 1] = 0.5 + np.abs(x[:, 1])
    x[17, 0] = 0.0
    y = rng.standard_normal(ROWS)
    y[17] = 9.0  # the row that a derivative of zero there vetoes
    return x, y


def _scan(trees, x, y, scale):
    ev = host.GpuEvaluator(np.ascontiguousarray(x.T, np.float32).reshape(-1), len(x), x.shape[1],
                           y.astype(np.float32))
    assert ev.set_fit_data(np.ascontiguousarray(x.T).reshape(-1), y)
    with np.errstate(all="ignore"):
        top = [float(np.max(np.abs(oracle.predict_flat(t, x) - y))) for t in trees]
    levels = [scale * v if math.isfinite(v) else 1.0 for v in top]
    runs = []
    for form in (lambda t: t, _on_the_general_kernel):
        outs, ms = ev.max_scan_batch([host.gpu_fit_plan(form(t)) for t in trees],
                                     coords=[0] * len(trees), levels=levels)
        assert ms >= 0
        runs.append(outs)
    ev.close()
    return levels, runs[0], runs[1]


def _agree(a, b, rel):
    if a.status != b.status or a.row != b.row:
        return False
    if a.status != 0:
        return True
    ends = zip((a.lo, a.hi), (b.lo, b.hi))
    return a.vmax == b.vmax and all(p == q if math.isinf(p) or math.isinf(q) else
                                    abs(p - q) <= rel * abs(q) for p, q in ends)


MAG = node(ABS, var(0))
LIMITS = {
    # Zero below a partial that is not finite, and above one.
    "sqrt at zero": node(SQRT, _line(1.2, MAG)),
    "sqrt of square at zero": node(SQRT, node(SQUARE, _line())),
    "square of sqrt at zero": node(SQUARE, node(SQRT, _line(1.2, MAG))),
    "power at zero": node(POW, _line(1.2, MAG), const(0.5)),
    "exponent": node(POW, var(1), _line(0.4)),
    # Partials that round to zero.
    "saturated": node(TANH, _scaled(_line(), 60.0)),
    "vanished": node(EXP, node(ADD, _scaled(_line(0.1), 1.0), const(-800.0))),
    # Products that leave the range, and come back.
    "subnormal on the way up": _scaled(_line(), 1e-200, 1e-113, 1e190),
    "zero on the way up": _scaled(_line(), 1e-200, 1e-140, 1e190),
    "infinite on the way up": _scaled(_line(1e-300), 1e160, 1e160, 1e-20),
    "subnormal on the way down": _scaled(_line(), 1e150, 1e-170, 1e-143),
    "zero on the way down": _scaled(_line(), 1e150, 1e-200, 1e-170),
    "infinite on the way down": _scaled(_line(), 1e-300, 1e160, 1e160),
    # The same through the two sides of a division.
    "numerator": node(DIV, _scaled(_line(), 1e-250), const(1e-11)),
    "denominator": _scaled(node(DIV, const(1e190), _line(1.2, var(1))), 1e-190),
    "numerator of a denominator": _scaled(
        node(DIV, const(1e200), node(MUL, _line(1.2, var(1)), const(1e150))), 1e-60),
}


@pytest.mark.parametrize("scale", [0.9, 1.3])
@pytest.mark.parametrize("name", list(LIMITS))
def test_derivatives_at_the_limits(name, scale):
    x, y = _rows()
    tree = LIMITS[name]
    print(f"order levels: {name}, scale {scale}", flush=True)
    (level,), (fast,), (general,) = _scan([tree], x, y, scale)
    assert _agree(fast, general, 1e-13), (fast, general)
    b = np.array([oracle.gradients(tree, r)[0][0] for r in x])
    vm, row, lo, hi, st = oracle.max_scan(oracle.predict_flat(tree, x) - y, b, level)
    assert (fast.status, fast.row) == (st, row)
    if st == 0:
        # The device's exp, tanh and pow are within a few ulp of the host's.
        assert fast.vmax == pytest.approx(vm, rel=1e-14)
        assert fast.lo == pytest.approx(lo, rel=1e-12) and fast.hi == pytest.approx(hi, rel=1e-12)


UNARY = [SIN, COS, TAN, EXP, SQRT, ABS, TANH, SIG, SQUARE, CUBE, NEG, GAUSS, SINH, COSH, ERF, ERFC]


def test_every_operator_under_every_other_on_both_routes():
    """u(v(c x)) over rows with zeros, ordinary and saturating values, and the
    binary operators on either side."""
    x, y = _rows()
    x[:, 0] = np.resize([0.0, 0.3, -0.3, 1.0, -1.0, 2.5, 6.0, 30.0, 1e-9, 300.0], ROWS)
    mag = [node(ABS, _line()) if u == SQRT else _line() for u in UNARY]
    inner = [node(u, a) for u, a in zip(UNARY, mag)]
    trees = [node(u, node(ABS, t) if u == SQRT else t) for u in UNARY for t in inner]
    for t in inner:
        trees += [node(DIV, t, var(1)), node(DIV, var(0), node(ADD, node(SQUARE, t), const(0.5))),
                  node(POW, node(ABS, t), const(1.7)), node(POW, var(1), t),
                  node(SUB, var(0), t), node(MUL, t, var(0))]
    print(f"order levels: {len(trees)} trees", flush=True)
    for scale in (0.9, 1.3):
        levels, fast, general = _scan(trees, x, y, scale)
        for t, a, b in zip(trees, fast, general):
            # tanh's 1 - f f is one fused operation in the general kernel and two
            # in the sweep: 2^-53 of 1, against a partial of 1e-7 and more in the
            # rows that set an end.
            rel = 1e-8 if "tanh" in str(t) else 1e-13
            assert _agree(a, b, rel), (str(t), scale, a, b)
