"""Work items of different sizes give the same bits: a candidate fitted by
itself (small items, RcSplit) and in a batch large enough for whole groups of
rows has the same constants, loss and status, for each arm that splits its
rows this way and at row counts on either side of a sub-tile's edge."""
import threading

import numpy as np
import pytest
import torch

from rcsr_hip import host
from rcsr_hip.expr import ADD, COS, MUL, SIN, SQUARE, SUB, const, node, var

pytestmark = pytest.mark.gpu

FIT = [node(ADD, node(MUL, const(0.8), node(SIN, node(MUL, const(1.3), var(0)))),
            node(MUL, const(0.3), var(1))),
       node(ADD, node(MUL, const(1.1), node(COS, var(0))), const(0.2))]
SHAPE = [node(ADD, node(MUL, const(1.4), node(SIN, node(MUL, const(1.2), var(0)))), const(-0.3))]
CURVE = [node(SUB, node(ADD, node(SQUARE, var(0)), node(MUL, const(0.9), node(SQUARE, var(1)))),
              const(1.1))]


def _evaluator(n):
    rng = np.random.default_rng(n)
    th = rng.uniform(0, 2 * np.pi, n)
    r = 1.0 + 0.02 * rng.standard_normal(n)
    x = np.stack([r * np.cos(th), r * np.sin(th)])
    y = np.sin(1.5 * x[0]) + 0.4 * x[1] + 0.05 * rng.standard_normal(n)
    ev = host.GpuEvaluator(x.astype(np.float32).reshape(-1), n, 2, y.astype(np.float32))
    assert ev.set_fit_data(x.reshape(-1), y)
    return ev


def _same(a, b):
    for o, p in zip(a, b):
        assert o.status == p.status and o.sse == p.sse and np.array_equal(o.c, p.c)


ARMS = {
    "squared": (FIT, lambda ev, plans: ev.fit_batch(plans, 6, 0)),
    "absolute": (FIT, lambda ev, plans: ev.fit_batch(plans, 6, 4)),
    "correlation": (SHAPE, lambda ev, plans: ev.fit_batch(plans, 6, 2,
                                                          gauge=[(0, 2)] * len(plans))),
    "implicit": (CURVE, lambda ev, plans: ev.implicit_fit_batch(plans, 3)),
}


# 8192 groups of up to 8192 rows in the full batch, against sub-tiles of 512 and
# 1024 rows for a candidate alone.
@pytest.mark.parametrize("n,copies", [(700, 8400), (8193, 4200), (20000, 2732)])
@pytest.mark.parametrize("arm", list(ARMS))
def test_a_candidate_alone_and_in_a_full_batch(arm, n, copies):
    trees, fit = ARMS[arm]
    ev = _evaluator(n)
    plans = [host.gpu_fit_plan(t) for t in trees]
    print(f"split: {arm}, {n} rows, {copies} copies", flush=True)
    alone, ms = fit(ev, plans)
    assert ms >= 0
    full, ms = fit(ev, plans * (copies // len(plans)))
    assert ms >= 0
    _same(full[:len(plans)], alone)
    _same(full[-len(plans):], alone)
    if arm == "squared":
        ev.set_fit_mode(host.FIT_MODE_FP64)
        alone, _ = fit(ev, plans)
        full, _ = fit(ev, plans * (copies // len(plans)))
        _same(full[-len(plans):], alone)
    ev.close()


@pytest.mark.parametrize("n", [511, 20000])
def test_implicit_scores_do_not_depend_on_the_batch(n):
    ev = _evaluator(n)
    plans = [host.gpu_fit_plan(t) for t in CURVE]
    alone, st, ms = ev.implicit_score_batch(plans)
    full, sf, mf = ev.implicit_score_batch(plans * 4200)
    assert ms >= 0 and mf >= 0 and not st.any() and not sf.any()
    assert np.all(full == alone[0])
    ev.close()


def test_implicit_scores_hold_two_sums_an_item():
    """8000 candidates x 8192 rows are 128 000 items: 2 MB of sums, where the
    fit's triangles would be 236 MB.  A second thread watches the free memory."""
    n, copies = 8192, 8000
    ev = _evaluator(n)
    plans = [host.gpu_fit_plan(CURVE[0])] * copies
    assert ev.implicit_score_batch(plans)[2] >= 0
    print(f"split: implicit score memory, {copies} x {n}", flush=True)
    before = torch.cuda.mem_get_info()[0]
    least, stop = [before], threading.Event()

    def watch():
        while not stop.is_set():
            least[0] = min(least[0], torch.cuda.mem_get_info()[0])

    t = threading.Thread(target=watch)
    t.start()
    score, st, ms = ev.implicit_score_batch(plans)
    stop.set()
    t.join()
    assert ms >= 0 and not st.any()
    assert before - least[0] <= 32 << 20
    ev.close()
