"""Work items of different sizes give the same bits: a candidate fitted by
itself (small items, RcSplit) and in a batch large enough for whole groups of
rows has the same constants, loss and status, for each arm that splits its
rows this way and at row counts on either side of a sub-tile's edge."""
import threading

import numpy as np
import pytest

from rcsr_hip import host, workloads
from rcsr_hip.expr import ADD, COS, LOG, MUL, SIN, SQUARE, SUB, const, node, var
from test_gpu_fit_tape import _basis, _tree

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


def _nested(levels):
    """A right-deep tree over two inputs: it keeps `levels` values below its top."""
    t = node(MUL, const(0.5), var(0))
    for i in range(levels):
        t = node(ADD if i % 2 else SUB, node(MUL, const(0.1 * (i + 1)), _basis(i, 2)), t)
    return t


# One program for every assembly kernel and value pass: 4-row streams with the
# tape in U, B and LDS (and their 2-row or general kernels with 2 rows per lane),
# 16 and 32 columns, and two programs outside the fit VM, of a small and of a
# large evaluation stack.
KERNELS = {"16 columns": FIT[0],
           "32 columns": workloads.structured_candidate(workloads.rng_for(3), 2, 18), "tape in B": _tree(16, 2, 0),
           "tape in LDS": _tree(20, 2, 2), "small stack": _nested(8), "large stack": _nested(11)}


@pytest.mark.parametrize("rows", [4, 2])
@pytest.mark.parametrize("metric", [0, 4])
@pytest.mark.parametrize("n", [8193, 20001])
def test_sub_tiles_and_whole_groups_of_every_kernel(n, metric, rows):
    """An item size of 8192 rows set by hand makes one item of each group: the
    kernels add its sub-tiles themselves."""
    ev = _evaluator(n)
    plans = [host.gpu_fit_plan(t) for t in KERNELS.values()]
    assert ev.set_tuning(host.TUNE_FIT_ROWS_PER_LANE, rows) == 0
    for mode in (host.FIT_MODE_MIXED, host.FIT_MODE_FP64) if metric == 0 else (host.FIT_MODE_MIXED,):
        ev.set_fit_mode(mode)
        print(f"split: {n} rows, metric {metric}, {rows} rows a lane, mode {mode}", flush=True)
        ev.set_tuning(host.TUNE_FIT_TILE_ROWS, 0)
        small, ms = ev.fit_batch(plans, 5, metric)
        assert ms >= 0 and all(np.isfinite(o.sse) for o in small)
        ev.set_tuning(host.TUNE_FIT_TILE_ROWS, 8192)
        whole, ms = ev.fit_batch(plans, 5, metric)
        assert ms >= 0
        _same(whole, small)
    ev.close()


@pytest.mark.parametrize("n", [8193, 20001])
def test_sub_tiles_and_whole_groups_of_the_correlation_kernels(n):
    ev = _evaluator(n)
    trees = [SHAPE[0], KERNELS["32 columns"], _nested(8), _nested(15)]
    plans = [host.gpu_fit_plan(t) for t in trees]
    small, ms = ev.fit_batch(plans, 5, 2)
    assert ms >= 0
    ev.set_tuning(host.TUNE_FIT_TILE_ROWS, 8192)
    whole, ms = ev.fit_batch(plans, 5, 2)
    assert ms >= 0
    _same(whole, small)
    ev.close()


# Relations for the sweeps beside the four-wide one: a guarded operator, and a
# stack beyond the register sweep's.
@pytest.mark.parametrize("n,copies", [(700, 8400), (8193, 4200)])
def test_implicit_relations_of_every_sweep(n, copies):
    trees = [node(SUB, node(ADD, node(SQUARE, var(0)), node(MUL, const(0.9), node(SQUARE, var(1)))),
                  node(SUB, const(1.1), node(LOG, node(ADD, const(3.0), var(0))))),
             node(ADD, _nested(10), node(SUB, node(SQUARE, var(1)), const(0.6)))]
    ev = _evaluator(n)
    plans = [host.gpu_fit_plan(t) for t in trees]
    print(f"split: implicit sweeps, {n} rows, {copies} copies", flush=True)
    alone, ms = ev.implicit_fit_batch(plans, 1)
    assert ms >= 0
    full, ms = ev.implicit_fit_batch(plans * (copies // len(plans)), 1)
    assert ms >= 0
    _same(full[:len(plans)], alone)
    _same(full[-len(plans):], alone)
    ev.close()


def test_implicit_scores_hold_two_sums_an_item(free_memory):
    """8000 candidates x 8192 rows are 128 000 items: 2 MB of sums, where the
    fit's triangles would be 236 MB.  A second thread watches the free memory."""
    n, copies = 8192, 8000
    ev = _evaluator(n)
    plans = [host.gpu_fit_plan(CURVE[0])] * copies
    assert ev.implicit_score_batch(plans)[2] >= 0
    print(f"split: implicit score memory, {copies} x {n}", flush=True)
    before = free_memory()
    least, stop = [before], threading.Event()

    def watch():
        while not stop.is_set():
            least[0] = min(least[0], free_memory())

    t = threading.Thread(target=watch)
    t.start()
    score, st, ms = ev.implicit_score_batch(plans)
    stop.set()
    t.join()
    assert ms >= 0 and not st.any()
    assert before - least[0] <= 32 << 20
    ev.close()
