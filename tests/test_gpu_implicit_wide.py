"""The implicit arm's four-wide sweep against the oracle and against the other
sweeps on the same relation: even and odd constant counts (the last sweep of a
Jacobian row is partly idle), one to three inputs, row counts around a step's
64 and 256 rows, weights with zeros, and undefined rows."""
import numpy as np
import pytest

import oracle
from rcsr_hip import host
from rcsr_hip.expr import ADD, COS, DIV, EXP, LOG, MUL, SIN, SQUARE, SUB, TANH, const, node, var

pytestmark = pytest.mark.gpu


def _terms(nv, k):
    """k - 1 coefficients and an offset near a closed curve (nv > 1)."""
    basis = [node(SQUARE, var(nv - 1)), node(SIN, var(0)), node(COS, var(nv - 1)),
             node(TANH, var(0)), node(EXP, node(MUL, const(0.1), var(nv - 1)))]
    terms = [node(SQUARE, var(0))]
    used = 1
    for i, b in enumerate(basis):
        cost = 2 if i == 4 else 1
        if used + cost > k:
            break
        terms.append(node(MUL, const(0.9 if i == 0 else 0.07 * (i + 1)), b))
        used += cost
    return terms


def _left(terms, c):
    t = terms[0]
    for u in terms[1:]:
        t = node(ADD, t, u)
    return node(SUB, t, const(c))


def _right(terms, c):
    t = node(SUB, terms[-1], const(c))
    for u in reversed(terms[:-1]):
        t = node(ADD, u, t)
    return t


def _rows(n, nv):
    rng = np.random.default_rng(17 * n + nv)
    th = rng.uniform(0, 2 * np.pi, n)
    r = 1.0 + 0.01 * rng.standard_normal(n)
    x = np.stack([r * np.cos(th), r * np.sin(th), rng.uniform(-1.5, 1.5, n)], 1)
    return np.ascontiguousarray(x[:, :nv])


def _evaluator(x, w=None):
    n, nv = x.shape
    ev = host.GpuEvaluator(np.ascontiguousarray(x.T, np.float32).reshape(-1), n, nv,
                           np.zeros(n, np.float32))
    assert ev.set_fit_data(np.ascontiguousarray(x.T).reshape(-1), np.zeros(n), w)
    return ev


@pytest.mark.parametrize("nv", [1, 2, 3])
@pytest.mark.parametrize("n", [1, 63, 65, 257, 900])
def test_scores_match_the_oracle(n, nv):
    x = _rows(n, nv)
    w = np.random.default_rng(n).uniform(0.1, 2.0, n)
    if n > 3:
        w[::3] = 0.0
    ev = _evaluator(x, w)
    trees = [_left(_terms(nv, k), 1.0) for k in (1, 2, 3, 5, 6)]
    trees.append(node(DIV, trees[1], node(ADD, const(2.0), node(SQUARE, var(0)))))
    plans = [host.gpu_fit_plan(t) for t in trees]
    print(f"implicit wide: {n} rows, {nv} inputs", flush=True)
    for metric in (0, 1):
        val, st, ms = ev.implicit_score_batch(plans, metric)
        assert ms >= 0 and not st.any()
        for v, t in zip(val, trees):
            # f64 rounding of a dozen operations a row
            assert v == pytest.approx(oracle.implicit_score(t, x, w, metric), rel=1e-12)
    ev.close()


@pytest.mark.parametrize("n", [65, 900])
@pytest.mark.parametrize("k", [2, 3, 4, 5, 6])
def test_fits_match_the_register_stack_sweep(k, n):
    x = _rows(n, 3)
    ev = _evaluator(x)
    terms = _terms(3, k - 1)
    # A guarded operator (of a positive argument) sends the second form to the
    # register-stack sweep; it adds log(1) = 0.
    guarded = node(ADD, _left(terms, 1.05), node(LOG, node(EXP, node(SUB, var(0), var(0)))))
    plans = [host.gpu_fit_plan(t) for t in (_left(terms, 1.05), guarded)]
    (a, b), ms = ev.implicit_fit_batch(plans, 4)
    assert ms >= 0 and a.status == b.status == 0
    # The same distances, bit for bit, in the same difference quotients.
    assert a.sse == b.sse and np.array_equal(a.c, b.c)
    (r,), ms = ev.implicit_fit_batch([host.gpu_fit_plan(_right(terms, 1.05))], 4)
    assert ms >= 0 and r.sse == pytest.approx(a.sse, rel=1e-6)
    ev.close()


def test_an_undefined_row_is_flagged():
    x = _rows(300, 2)
    x[131] = 0.0                       # the gradient of x0^2 + x1^2 - 1 vanishes
    ev = _evaluator(x)
    t = node(SUB, node(ADD, node(SQUARE, var(0)), node(MUL, const(1.0), node(SQUARE, var(1)))),
             const(1.0))
    plans = [host.gpu_fit_plan(t)]
    val, st, ms = ev.implicit_score_batch(plans)
    assert ms >= 0 and st[0] == 2 and np.isinf(val[0])
    (o,), ms = ev.implicit_fit_batch(plans, 2)
    assert ms >= 0 and o.status == 7
    ev.close()
