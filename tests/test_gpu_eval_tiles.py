"""The evaluator's row tiles over small and odd tables, the allocation-free
entry point where its partial sums take several parts, the one-pass
correlation score, and the rare operators' shared call, against f64
reductions of the device's own predictions."""
import numpy as np
import pytest

from rcsr_hip import host, lib
from rcsr_hip.expr import (ADD, ATAN2, CUBE, DIV, ERF, IF, LOG, MAX, MOD, MUL, POW, SIN, SQRT, SUB,
                           TAN, TANH, const, node, var)

pytestmark = pytest.mark.gpu

TREES = [node(ADD, node(MUL, const(1.3), var(0)), const(0.2)),
         node(TANH, node(ADD, var(0), node(SIN, var(1)))),
         node(ERF, node(CUBE, var(0))),
         node(ADD, node(TAN, var(0)), node(SQRT, node(MUL, var(1), var(1)))),
         node(MAX, node(MOD, var(0), const(0.7)), node(ATAN2, var(1), var(0))),
         node(POW, node(MUL, var(0), var(0)), const(0.6)),
         node(IF, var(0), node(TANH, var(1)), node(DIV, var(0), const(3.0))),
         node(ADD, const(2.0e4), var(0))]


def _evaluator(n):
    rng = np.random.default_rng(n)
    x = rng.standard_normal((2, n)).astype(np.float32)
    y = (x[0] + 0.3 * rng.standard_normal(n)).astype(np.float32)
    return y, host.GpuEvaluator(x.reshape(-1), n, 2, y)


def _words(trees):
    pop = host.Population()
    assert all(pop.add(t) for t in trees)
    return pop.arrays()


@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 1000, 4096, 4097, 5000, 32768, 32769])
def test_losses_and_correlation_scores_of_every_tile_size(n):
    y, ev = _evaluator(n)
    prog, off = _words(TREES)
    print(f"eval tiles: {n} rows", flush=True)
    pred = ev.predict_words(prog, off)
    assert np.isfinite(pred).all()
    out, ms = ev.eval_words(prog, off, 0)
    rr = (pred - y).astype(np.float32)
    want = np.sum((rr * rr).astype(np.float64), 1)
    assert ms >= 0 and np.allclose(out, want, rtol=1.2e-7, atol=0)   # one f32 rounding
    p, dy = pred.astype(np.float64), y.astype(np.float64) - y.astype(np.float64).mean()
    dp = p - p.mean(1, keepdims=True)
    ss, yy = np.sum(dp * dp, 1), np.sum(dy * dy)
    rho = np.zeros(len(TREES)) if n == 1 else (dp @ dy) / np.sqrt(ss * yy)
    for kind, want in ((5, 1.0 - np.abs(rho)), (6, 1.0 - rho)):
        score, st, ms = ev.score_words(prog, off, kind)
        assert ms >= 0 and not st.any()
        # f64 sums of n terms on both sides; the last program's mean is 2e4 of its
        # spread, which costs the f64 mean that many of its digits.
        assert np.allclose(score, want, rtol=0, atol=1e-11)
    ev.close()


def test_correlation_flags_a_row_that_is_not_finite_wherever_it_is():
    n = 9000
    x = np.ones((1, n), np.float32)
    for bad in (0, 1, 4095, 4096, n - 1):
        x[0, bad] = -1.0
        ev = host.GpuEvaluator(x.reshape(-1), n, 1, np.arange(n, dtype=np.float32))
        prog, off = _words([node(LOG, var(0)), var(0)])
        score, st, ms = ev.score_words(prog, off, 5)
        assert ms >= 0 and list(st) == [2, 0] and np.isinf(score[0]) and np.isfinite(score[1])
        x[0, bad] = 1.0
        ev.close()


# The first row's prediction is far from all others, over tiles of the built-in
# size and of the largest that can be set: the moments about a pivot near it
# would lose as many digits as a tile has rows.
@pytest.mark.parametrize("n,tile", [(300, 0), (4096, 4096), (60000, 0), (1 << 20, 1 << 20)])
@pytest.mark.parametrize("outliers", [1, 40])
def test_correlation_of_predictions_with_an_outlier_in_the_first_row(n, tile, outliers):
    rng = np.random.default_rng(n)
    x = rng.standard_normal((1, n)).astype(np.float32)
    y = (x[0] + 0.3 * rng.standard_normal(n)).astype(np.float32)
    x[0, :outliers] = 1e6
    ev = host.GpuEvaluator(x.reshape(-1), n, 1, y)
    assert ev.set_tuning(host.TUNE_EVAL_TILE_ROWS, tile) == 0
    prog, off = _words([var(0)])
    print(f"correlation with {outliers} outliers: {n} rows, tile {tile}", flush=True)
    p, q = x[0].astype(np.longdouble), y.astype(np.longdouble)
    dp, dy = p - p.mean(), q - q.mean()
    rho = float(np.sum(dp * dy) / np.sqrt(np.sum(dp * dp) * np.sum(dy * dy)))
    score, st, ms = ev.score_words(prog, off, 6)
    assert ms >= 0 and not st.any()
    # 1 - r of an r near 0: sums of n / 64 terms a lane, their roundings of 2^-53
    # adding up like a random walk, and up to 16 times that in the tile that the
    # outliers are in.
    assert abs(score[0] - (1.0 - rho)) <= 16 * 2.0 ** -53 * max(np.sqrt(n / 64), 8) * max(rho, 1e-3) + 4e-16
    ev.close()


def test_only_the_scores_with_further_sums_hold_memory_for_them(free_memory):
    n, copies = 4096, 7500
    y, ev = _evaluator(n)
    prog, off = _words(TREES)
    lens = np.tile(np.diff(off), copies)
    big = np.tile(prog, copies).astype(np.uint32)
    boff = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    assert ev.eval_words(big, boff, 0)[1] >= 0    # grows the sums that every score has too
    print(f"score memory: {len(boff) - 1} programs x {n} rows", flush=True)
    free = free_memory()
    score, st, ms = ev.score_words(big, boff, 0)
    assert ms >= 0
    # 960 000 items: 8 bytes each for a second sum would be 7.7 MB; the values and
    # statuses of the call are 0.7 MB.
    assert free - free_memory() <= 4 << 20
    ev.close()


def test_static_evaluation_in_several_parts():
    n, copies = 4000, 19000
    y, ev = _evaluator(n)
    prog, off = _words(TREES)
    lens = np.tile(np.diff(off), copies)
    big = np.tile(prog, copies).astype(np.uint32)
    boff = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    nprog = len(boff) - 1
    out = np.zeros(nprog, np.float32)
    print(f"static evaluation: {nprog} programs x {n} rows", flush=True)
    ms = ev._L.rc_eval_static(ev.ctx, lib.ptr(big, lib.u32p), lib.ptr(boff, lib.u32p), nprog,
                              lib.ptr(out, lib.f32p), 0)
    assert ms >= 0
    want, ms = ev.eval_words(prog, off, 0)
    assert ms >= 0
    assert np.array_equal(out.reshape(copies, -1).view(np.uint32),
                          np.tile(want, (copies, 1)).view(np.uint32))
    ev.close()
