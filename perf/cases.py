"""The work that a symbolic-regression search has the device arm do, as timed
cases: one dict of plain values per case, inputs made from a seed, one pass
through the public entry points, and the same pass in 64-bit torch.

A search alternates between scoring whole generations of programs and
fitting the constants of the promising ones, over anything from a thousand
rows (one island of a small table) to a quarter of a million or a million.
The kinds below are those calls:

  eval      loss sums of a batch of programs (rc_set_programs + rc_eval)
  score     a native score objective of a batch (rc_score_batch)
  pool      one generation on the resident pool: device variation, then the
            children's losses (rc_pool_vary + rc_pool_eval)
  fit       batched LM / IRLS constant fitting (rc_fit_batch, metrics 0, 1, 4)
  hetero    one fit batch over islands with row sets and metrics of their own
            (rc_fit_batch_hetero)
  corr      the correlation fit objective with a gauge pair (metric 2)
  implicit  implicit relations (rc_implicit_fit_batch, rc_implicit_score_batch)
  order     exact order, rank and maximum statistics of candidate residuals
            (rc_order_stat_score_batch, rc_rank_score_batch, rc_max_scan_batch)

Programs are nested tuples (operator name, children ...), ("c", slot) for a
constant and ("x", column) for an input; the framework's trees are made from
them in prepare(), and exact() evaluates the tuples themselves.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "the-rule-and-compass_amd"))

from rcsr_hip import expr, host, lib  # noqa: E402

OPS = {"+": expr.ADD, "-": expr.SUB, "*": expr.MUL, "/": expr.DIV, "sin": expr.SIN,
       "cos": expr.COS, "exp": expr.EXP, "log": expr.LOG, "tanh": expr.TANH,
       "square": expr.SQUARE}


# ---- cases ------------------------------------------------------------------

def listed():
    return [
        # One island's offspring on a small table: every launch counts.
        {"name": "eval-island", "kind": "eval", "rows": 1000, "cols": 2, "programs": 200,
         "nodes": 31, "loss": 0},
        # A wide generation over a large table, the throughput end.
        {"name": "eval-generation", "kind": "eval", "rows": 1048576, "cols": 5, "programs": 4096,
         "nodes": 60, "loss": 0},
        # Selection by correlation over a mid-sized table of odd length; some
        # programs are undefined on some rows.
        {"name": "score-correlation", "kind": "score", "rows": 154001, "cols": 5, "programs": 512,
         "nodes": 40, "score": 5},
        # One generation of the flat engine kept on the device.
        {"name": "pool-generation", "kind": "pool", "rows": 5000, "islands": 16, "pop": 256,
         "nodes": 30},
        # Fits of one island's best on a small table, eight iterations.
        {"name": "fit-island", "kind": "fit", "rows": 1000, "candidates": 200, "kmin": 1,
         "kmax": 4, "iters": 8, "metric": 0},
        # A few promoted candidates, absolute error (IRLS), odd row count.
        {"name": "fit-absolute", "kind": "fit", "rows": 100003, "candidates": 64, "kmin": 1,
         "kmax": 16, "iters": 8, "metric": 4},
        # The large fit: 1 to 18 constants, a quarter of a million rows.
        {"name": "fit-wide", "kind": "fit", "rows": 262144, "candidates": 1024, "kmin": 1,
         "kmax": 18, "iters": 30, "metric": 0},
        # Islands of very different sizes and two metrics in one batch.
        {"name": "fit-islands", "kind": "hetero", "rows": 400000, "rmin": 512, "islands": 8,
         "candidates": 64, "kmin": 1, "kmax": 18, "iters": 8},
        # Correlation objective: the shape is fitted, the affine pair frozen.
        {"name": "fit-correlation", "kind": "corr", "rows": 50021, "candidates": 128, "kmin": 3,
         "kmax": 12, "iters": 12},
        # Implicit relations on noisy points of a closed curve.
        {"name": "implicit-fit", "kind": "implicit", "rows": 65537, "candidates": 128, "kmin": 2,
         "kmax": 7, "iters": 8},
        # Median absolute error of candidates under several constant vectors.
        {"name": "order-median", "kind": "order", "rows": 262144, "candidates": 64, "trials": 4,
         "what": "median"},
        # Largest error and the step along a constant that keeps a level.
        {"name": "order-maximum", "kind": "order", "rows": 100003, "candidates": 64, "trials": 4,
         "what": "level"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same calls, sizes spread over their logarithm."""
    kind = rng.choice(["eval", "eval", "score", "pool", "fit", "fit", "hetero", "corr",
                       "implicit", "order", "order"])
    if kind == "eval":
        rows, progs = _log(rng, 300, 1000000), _log(rng, 16, 4096)
        return {"kind": kind, "rows": rows, "cols": rng.randint(1, 6), "programs": progs,
                "nodes": rng.randint(11, 60), "loss": rng.choice([0, 0, 1, 4])}
    if kind == "score":
        return {"kind": kind, "rows": _log(rng, 1000, 500000), "cols": rng.randint(1, 6),
                "programs": _log(rng, 32, 1024), "nodes": rng.randint(11, 50),
                "score": rng.choice([0, 1, 2, 4, 5])}
    if kind == "pool":
        return {"kind": kind, "rows": _log(rng, 500, 50000), "islands": rng.randint(2, 20),
                "pop": _log(rng, 64, 512), "nodes": rng.randint(15, 40)}
    if kind == "fit":
        kmin = rng.randint(1, 4)
        rows, cands = _log(rng, 600, 262144), _log(rng, 24, 900)
        metric = rng.choice([0, 0, 0, 1, 4])
        cands = cands if metric == 0 else min(cands, 300)
        return {"kind": kind, "rows": rows, "candidates": cands, "kmin": kmin,
                "kmax": rng.randint(kmin, 18), "iters": rng.choice([8, 12, 30]), "metric": metric}
    if kind == "hetero":
        return {"kind": kind, "rows": _log(rng, 20000, 600000), "rmin": rng.randint(500, 3000),
                "islands": rng.randint(2, 10), "candidates": _log(rng, 16, 96), "kmin": 1,
                "kmax": rng.randint(4, 18), "iters": rng.choice([8, 12])}
    if kind == "corr":
        return {"kind": kind, "rows": _log(rng, 2000, 150000), "candidates": _log(rng, 24, 200),
                "kmin": 3, "kmax": rng.randint(4, 14), "iters": rng.choice([12, 20, 30])}
    if kind == "implicit":
        return {"kind": kind, "rows": _log(rng, 4000, 100000), "candidates": _log(rng, 24, 128),
                "kmin": 2, "kmax": rng.randint(3, 7), "iters": rng.choice([0, 8, 8])}
    return {"kind": kind, "rows": _log(rng, 1000, 262144), "candidates": rng.randint(8, 64),
            "trials": rng.choice([1, 2, 4]),
            "what": rng.choice(["median", "quartiles", "ranks", "maximum", "level"])}


# ---- programs ---------------------------------------------------------------

def _bounded(rng, cols, size):
    """A random program of about `size` nodes, defined and moderate on every
    row: divisors and log arguments are 1.5 + square, exp sees a bounded
    argument."""
    if size <= 1:
        if rng.random() < 0.3:
            return ("k", float(np.float32(rng.standard_normal())))
        return ("x", int(rng.integers(cols)))
    if size == 2 or rng.random() < 0.3:
        op = ("sin", "cos", "tanh", "exp", "log")[int(rng.integers(5))]
        if op == "exp":
            return ("exp", ("sin", _bounded(rng, cols, size - 2)))
        if op == "log":
            return ("log", ("+", ("k", 1.5), ("square", _bounded(rng, cols, size - 4))))
        return (op, _bounded(rng, cols, size - 1))
    left = int(rng.integers(1, size - 1))
    op = "+-*/"[int(rng.integers(4))]
    a, b = _bounded(rng, cols, left), _bounded(rng, cols, size - 1 - left)
    if op == "/":
        b = ("+", ("k", 1.5), ("square", b))
    elif op == "*" and left > 8:
        b = ("tanh", b)
    return (op, a, b)


def _programs(case, rng):
    out = []
    for i in range(case["programs"]):
        t = _bounded(rng, case["cols"], int(rng.integers(3, case["nodes"] + 1)))
        if case["kind"] == "score" and i % 25 == 7:
            t = ("+", t, ("log", ("x", 0)))  # undefined where the column is negative
        out.append(t)
    return out


# Terms of the target that the fitted candidates share, with the true values
# of their constants: one for each way of being odd or even in the inputs, so
# that a candidate without some of them still has an optimum of its own.
TERMS = [
    (("*", ("c",), ("*", ("exp", ("*", ("c",), ("square", ("x", 0)))), ("x", 0))), (1.7, -0.7)),
    (("*", ("c",), ("*", ("cos", ("*", ("c",), ("x", 1))), ("x", 1))), (0.8, 1.4)),
    (("*", ("c",), ("tanh", ("*", ("c",), ("x", 2)))), (1.2, 1.1)),
    (("*", ("c",), ("sin", ("*", ("c",), ("*", ("x", 0), ("x", 1))))), (1.0, 1.1)),
    (("*", ("c",), ("/", ("*", ("x", 0), ("x", 2)), ("+", ("c",), ("square", ("x", 0))))),
     (1.4, 0.8)),
    (("*", ("c",), ("tanh", ("*", ("c",), ("*", ("x", 1), ("x", 2))))), (0.9, 1.2)),
]
# Terms that are linear in their one constant, and the term above that each
# would take the place of (a candidate has one or the other), or None.
LINEAR = [(("square", ("x", 0)), None), (("square", ("x", 1)), None), (("square", ("x", 2)), None),
          (("square", ("*", ("x", 0), ("x", 1))), None), (("cos", ("*", ("x", 0), ("x", 2))), None),
          (("square", ("*", ("x", 1), ("x", 2))), None),
          (("*", ("x", 0), ("*", ("x", 1), ("x", 2))), None),
          (("*", ("x", 0), ("square", ("x", 1))), None),
          (("*", ("x", 2), ("square", ("x", 0))), None),
          (("sin", ("*", ("x", 1), ("square", ("x", 2)))), None),
          (("cos", ("+", ("x", 1), ("x", 2))), None),
          (("x", 0), 0), (("x", 1), 1), (("x", 2), 2), (("*", ("x", 0), ("x", 1)), 3),
          (("*", ("x", 0), ("x", 2)), 4), (("*", ("x", 1), ("x", 2)), 5)]
OFFSET = 0.25


def _number(t, start):
    """Number the constants of a tuple tree in the order of its leaves."""
    if t[0] == "c":
        return ("c", start), start + 1
    if t[0] in ("x", "k"):
        return t, start
    kids = []
    for k in t[1:]:
        k, start = _number(k, start)
        kids.append(k)
    return (t[0], *kids), start


def _sum(terms):
    t = terms[0]
    for u in terms[1:]:
        t = ("+", t, u)
    return t


def _candidate(rng, k):
    """A sum of terms with exactly k constants and their start values: the
    nonlinear ones within some 15% of what generated the rows, as those of an
    offspring of a fitted parent are, the linear ones anywhere."""
    while True:
        terms, c0, left, used = [], [], k, set()
        for i in rng.permutation(len(TERMS)):
            t, true = TERMS[i]
            if len(true) <= left and rng.random() < 0.6:
                terms.append(t)
                c0 += [v * (1.0 + 0.15 * float(np.clip(rng.standard_normal(), -1.5, 1.5)))
                       for v in true]
                left -= len(true)
                used.add(i)
        linear = _linear(rng, used) + [("c",)]
        if left <= len(linear):
            # The plain offset takes the last place in half of them.
            terms += linear[:left] if rng.random() < 0.5 else linear[len(linear) - left:]
            c0 += [float(v) for v in rng.standard_normal(left)]
            tree = _number(_sum(terms), 0)[0]
            if _nodes(tree) <= host.GPU_FIT_MAX_NODES:
                return tree, c0


def _linear(rng, used):
    """The linear terms beside the terms `used`, in some order."""
    return [("*", ("c",), LINEAR[i][0]) for i in rng.permutation(len(LINEAR))
            if LINEAR[i][1] not in used]


def _nodes(t):
    return 1 if t[0] in ("c", "x", "k") else 1 + sum(_nodes(u) for u in t[1:])


def _shaped(rng, k):
    """a * shape + b with k constants in all for the correlation objective,
    near its optimum; the shape's first term has no scale of its own, which a
    would repeat."""
    while True:
        i = int(rng.integers(len(TERMS)))
        t, true = TERMS[i]
        first, start = t[2], [v * (1.0 + 0.1 * float(rng.uniform(-1, 1))) for v in true[1:]]
        left = k - 2 - len(start)
        if left >= 0:
            break
    terms, c0, used = [first], start, {i}
    for j in rng.permutation(len(TERMS)):
        t, at = TERMS[j]
        if j not in used and len(at) <= left and rng.random() < 0.8:
            terms.append(t)
            scale = (at[0] / true[0],) + at[1:]
            c0 += [v * (1.0 + 0.1 * float(rng.uniform(-1, 1))) for v in scale]
            left -= len(at)
            used.add(j)
    terms += _linear(rng, set(range(len(TERMS))))[:left]
    c0 += [0.02 * float(v) for v in rng.standard_normal(left)]
    tree = _number(("+", ("*", ("c",), _sum(terms)), ("c",)), 0)[0]
    return tree, [1.5 * true[0]] + c0 + [float(rng.standard_normal())]


IMPLICIT_BASIS = [("square", ("x", 1)), ("*", ("x", 0), ("x", 1)), ("x", 0), ("x", 1), ("x", 2),
                  ("sin", ("x", 0))]


def _relation(rng, k):
    """x0^2 + c x1^2 + ... - c' with k constants, near the curve of the rows."""
    terms, c0 = [("square", ("x", 0)), ("*", ("c",), IMPLICIT_BASIS[0])], []
    c0.append(1.0 + 0.1 * float(rng.uniform(-1, 1)))
    for j in 1 + rng.permutation(len(IMPLICIT_BASIS) - 1)[:k - 2]:
        terms.append(("*", ("c",), IMPLICIT_BASIS[j]))
        c0.append(0.1 * float(rng.uniform(-1, 1)))
    c0.append(1.0 + 0.1 * float(rng.uniform(-1, 1)))
    return _number(("-", _sum(terms), ("c",)), 0)[0], c0


def _tree(t, c):
    """The framework's tree of a tuple program with constants c."""
    if t[0] == "c":
        return expr.const(c[t[1]])
    if t[0] == "k":
        return expr.const(t[1])
    if t[0] == "x":
        return expr.var(t[1])
    return expr.node(OPS[t[0]], *(_tree(k, c) for k in t[1:]))


# ---- rows -------------------------------------------------------------------

def _table(case, rng):
    """Standard normal columns and target of an evaluation, as f32."""
    x = rng.standard_normal((case["cols"], case["rows"]), dtype=np.float32)
    return x, rng.standard_normal(case["rows"], dtype=np.float32)


def _target(x):
    y = np.full(x.shape[1], OFFSET)
    for t, true in TERMS:
        y += _np(_number(t, 0)[0], x, true)
    return y


def _np(t, x, c):
    if t[0] == "c":
        return c[t[1]]
    if t[0] == "k":
        return t[1]
    if t[0] == "x":
        return x[t[1]]
    k = [_np(u, x, c) for u in t[1:]]
    return {"+": lambda a, b: a + b, "-": lambda a, b: a - b, "*": lambda a, b: a * b,
            "/": lambda a, b: a / b, "sin": np.sin, "cos": np.cos, "exp": np.exp, "log": np.log,
            "tanh": np.tanh, "square": np.square}[t[0]](*k)


def _fit_rows(rng, rows, outliers):
    """Three inputs, uniform; a target of all the terms with small noise, and
    one row in a hundred far off where the metric is a robust one."""
    x = rng.uniform(-2.0, 2.0, size=(3, rows))
    y = _target(x) + 0.05 * rng.standard_normal(rows)
    if outliers:
        far = rng.random(rows) < 0.01
        y[far] += 3.0 * rng.standard_cauchy(int(far.sum())).clip(-50.0, 50.0)
    return x, y


def _curve(rng, rows):
    """Noisy points of a circle and a column that has no part in it."""
    th = rng.uniform(0.0, 2.0 * np.pi, rows)
    r = 1.0 + 0.01 * rng.standard_normal(rows)
    return np.stack([r * np.cos(th), r * np.sin(th), rng.uniform(-1.5, 1.5, rows)])


# ---- inputs of a case, without the framework ------------------------------------

def _inputs(case, seed):
    rng = np.random.default_rng([seed, 97])
    kind = case["kind"]
    d = {}
    if kind in ("eval", "score"):
        d["x"], d["y"] = _table(case, rng)
        d["trees"] = _programs(case, rng)
        return d
    if kind == "pool":
        d["x"] = rng.uniform(-2.0, 2.0, size=(2, case["rows"])).astype(np.float32)
        d["y"] = (np.sin(d["x"][0]) + 0.5 * d["x"][1] ** 2).astype(np.float32)
        n = case["islands"] * case["pop"]
        d["trees"] = [_bounded(rng, 2, int(rng.integers(3, max(4, case["nodes"] // 2))))
                      for _ in range(n)]
        d["err"] = rng.exponential(1.0, n)
        d["seed"] = int(rng.integers(1 << 30))
        return d

    def ks():  # every count alike, so that a case's outputs have one shape
        return case["kmin"] + np.arange(case["candidates"]) % (case["kmax"] + 1 - case["kmin"])
    if kind == "fit":
        d["x"], d["y"] = _fit_rows(rng, case["rows"], case["metric"] != 0)
        d["cands"] = [_candidate(rng, int(k)) for k in ks()]
    elif kind == "hetero":
        sizes = np.exp(rng.uniform(np.log(case["rmin"]), np.log(case["rows"]),
                                   case["islands"])).astype(int)
        sizes[0] = case["rows"]
        d["sets"] = [_fit_rows(rng, int(s), True) for s in sizes]
        d["cands"], d["set"], d["metric"] = [], [], []
        for i in range(case["islands"]):
            d["cands"] += [_candidate(rng, int(k)) for k in ks()]
            d["set"] += [i] * case["candidates"]
            d["metric"] += [int(m) for m in rng.choice([0, 4], case["candidates"])]
    elif kind == "corr":
        d["x"], d["y"] = _fit_rows(rng, case["rows"], False)
        d["cands"] = [_shaped(rng, int(k)) for k in ks()]
    elif kind == "implicit":
        d["x"] = _curve(rng, case["rows"])
        d["y"] = np.zeros(case["rows"])
        d["cands"] = [_relation(rng, int(k)) for k in ks()]
    else:
        d["x"], d["y"] = _fit_rows(rng, case["rows"], False)
        d["cands"] = [_candidate(rng, 1 + i % 18) for i in range(case["candidates"])]
        kmax = max(len(c) for _, c in d["cands"])
        d["c"] = np.zeros((case["candidates"] * case["trials"], kmax))
        for i, (_, c) in enumerate(d["cands"]):
            for t in range(case["trials"]):
                step = 0.02 * t * rng.standard_normal(len(c))
                d["c"][i * case["trials"] + t, :len(c)] = np.asarray(c) * (1.0 + step)
    return d


# ---- the framework ------------------------------------------------------------

def _evaluator(x, y, exact_rows=True):
    ev = host.GpuEvaluator(np.asarray(x, np.float32).reshape(-1), x.shape[1], x.shape[0],
                           np.asarray(y, np.float32))
    if exact_rows and not ev.set_fit_data(np.asarray(x, np.float64).reshape(-1),
                                          np.asarray(y, np.float64)):
        raise RuntimeError("set_fit_data failed")
    return ev


def _plans(cands):
    plans = [host.gpu_fit_plan(_tree(t, c)) for t, c in cands]
    if any(p is None for p in plans):
        raise RuntimeError("a candidate has no fit plan")
    return plans


POOL_WIDTH = 64
POOL_OPS = np.array([[expr.ADD, 2], [expr.SUB, 2], [expr.MUL, 2], [expr.DIV, 2], [expr.SIN, 1],
                     [expr.COS, 1], [expr.EXP, 1], [expr.LOG, 1]], np.uint32).reshape(-1)


def prepare(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    s = {"case": case}
    if kind in ("eval", "score", "pool"):
        s["ev"] = _evaluator(d["x"], d["y"], False)
        words = [host.compile_program(_tree(t, ())) for t in d["trees"]]
        if kind == "pool":
            blank = np.full((len(words), POOL_WIDTH), expr.HALT, np.uint32)
            for i, w in enumerate(words):
                if len(w) > POOL_WIDTH:  # rare: such a slot starts as one column
                    w = host.compile_program(expr.var(i % 2))
                blank[i, :len(w)] = w
            ev = s["ev"]
            if (ev._L.rc_pool_reserve(ev.ctx, len(words), POOL_WIDTH) != 0 or
                    ev._L.rc_pool_upload(ev.ctx, 0, lib.ptr(blank.reshape(-1), lib.u32p),
                                         len(words)) != 0):
                raise RuntimeError("pool upload failed")
            s["err"], s["seed"] = d["err"], d["seed"]
            return s
        s["prog"] = np.concatenate(words)
        s["off"] = np.concatenate([[0], np.cumsum([len(w) for w in words])]).astype(np.uint32)
        return s
    if kind == "hetero":
        x, y = d["sets"][0]
        s["ev"] = ev = _evaluator(x, y)
        for x, y in d["sets"][1:]:
            if ev.add_rows(x.astype(np.float32).reshape(-1), x.shape[1], 3, y.astype(np.float32),
                           x.reshape(-1), y) < 0:
                raise RuntimeError("add_rows failed")
        s["set"], s["metric"] = d["set"], d["metric"]
    else:
        s["ev"] = _evaluator(d["x"], d["y"])
    s["plans"] = _plans(d["cands"])
    if kind == "corr":
        s["gauge"] = [(0, len(c) - 1) for _, c in d["cands"]]
    if kind == "order":
        s["c"] = d["c"]
        if case["what"] == "level":
            s["coords"] = [0] * len(d["c"])
            s["levels"] = [LEVEL] * len(d["c"])
    return s


LEVEL = 12.0


def _fitted(outs, ms):
    if ms < 0:
        raise RuntimeError("the fit failed")
    return {"c": np.concatenate([o.c for o in outs]), "loss": np.array([o.sse for o in outs]),
            "status": np.array([o.status for o in outs], np.int32)}


def run(s):
    case, ev = s["case"], s["ev"]
    kind = case["kind"]
    if kind == "eval":
        out, ms = ev.eval_words(s["prog"], s["off"], case["loss"])
        if ms < 0:
            raise RuntimeError("the evaluation failed")
        return {"loss": out}
    if kind == "score":
        out, status, ms = ev.score_words(s["prog"], s["off"], case["score"])
        if ms < 0:
            raise RuntimeError("the score failed")
        return {"score": out, "status": status}
    if kind == "pool":
        return _generation(s)
    if kind == "fit":
        return _fitted(*ev.fit_batch(s["plans"], case["iters"], case["metric"]))
    if kind == "hetero":
        return _fitted(*ev.fit_batch_hetero(s["plans"], s["set"], s["metric"], case["iters"]))
    if kind == "corr":
        return _fitted(*ev.fit_batch(s["plans"], case["iters"], 2, gauge=s["gauge"]))
    if kind == "implicit":
        if case["iters"] > 0:
            return _fitted(*ev.implicit_fit_batch(s["plans"], case["iters"]))
        out, status, ms = ev.implicit_score_batch(s["plans"], 0)
        if ms < 0:
            raise RuntimeError("the implicit score failed")
        return {"score": out, "status": status}
    what, trials = case["what"], case["trials"]
    if what in ("median", "quartiles"):
        out, status, ms = ev.order_stat_batch(s["plans"], 0 if what == "median" else 1, s["c"],
                                              trials)
        if ms < 0:
            raise RuntimeError("the order statistic failed")
        return {"value": out, "status": status}
    if what == "ranks":
        sums, bb, status, ms = ev.rank_score_batch(s["plans"], s["c"], trials)
        if ms < 0:
            raise RuntimeError("the rank sums failed")
        return {"sums": np.array(sums, np.float64), "target": float(bb), "status": status}
    out, ms = ev.max_scan_batch(s["plans"], s["c"], trials, s.get("coords"), s.get("levels"))
    if ms < 0:
        raise RuntimeError("the maximum scan failed")
    res = {"max": np.array([o.vmax for o in out]), "row": np.array([o.row for o in out], np.int32)}
    if what == "level":
        res["lo"] = np.array([o.lo for o in out])
        res["hi"] = np.array([o.hi for o in out])
    return res


def _generation(s):
    case, ev = s["case"], s["ev"]
    n = case["islands"] * case["pop"]
    length, cost = np.zeros(n, np.uint16), np.zeros(n, np.uint16)
    key, err, loss = np.zeros(n, np.uint64), np.zeros(n), np.zeros(n, np.float32)
    rc = ev._L.rc_pool_vary(ev.ctx, 0, case["islands"], case["pop"], s["seed"], 1, case["nodes"],
                            2, 3, 1, lib.ptr(POOL_OPS, lib.u32p), len(POOL_OPS) // 2,
                            lib.ptr(s["err"], lib.f64p), None, lib.ptr(length, lib.u16p),
                            lib.ptr(cost, lib.u16p), lib.ptr(key, lib.u64p),
                            lib.ptr(err, lib.f64p))
    if rc != 0 or ev._L.rc_pool_eval(ev.ctx, 1, n, POOL_WIDTH, lib.ptr(loss, lib.f32p), 0) < 0:
        raise RuntimeError("the generation failed")
    return {"length": length.astype(np.int32), "cost": cost.astype(np.int32),
            "hash": key.view(np.int64), "error": err, "loss": loss}


# ---- what a pass cannot do without ------------------------------------------------

def _flops(t):
    """Arithmetic of one row of a program: one for each plain operator, twenty
    for each transcendental one."""
    if t[0] in ("c", "k", "x"):
        return 0
    own = 20 if t[0] in ("sin", "cos", "exp", "log", "tanh") else 1
    return own + sum(_flops(k) for k in t[1:])


def work(case):
    kind = case["kind"]
    if kind in ("eval", "score", "pool"):
        progs = case.get("programs") or case["islands"] * case["pop"]
        small = dict(case, programs=min(progs, 64), cols=case.get("cols", 2))
        mean = np.mean([_flops(t) for t in _programs(small, np.random.default_rng(5))])
        words = 0.6 * case["nodes"] * 4.0
        return {"bytes": 4.0 * case["rows"] * (small["cols"] + 1) + progs * (words + 8.0),
                "flops": float(progs * case["rows"] * (mean + 3.0))}
    # A fit that starts near its optimum cannot do without some four
    # assemblies (value, gradient, k x k products) and as many losses;
    # a correlation or implicit fit is counted alike.
    rng = np.random.default_rng(5)
    make = {"corr": _shaped, "implicit": _relation}.get(kind, _candidate)
    kmin, kmax = case.get("kmin", 1), case.get("kmax", 18)
    sample = [make(rng, int(k)) for k in rng.integers(kmin, kmax + 1, 32)]
    value = np.mean([_flops(t) for t, _ in sample])
    k = np.mean([float(len(c)) ** 2 + len(c) for _, c in sample])
    cands, rows = float(case["candidates"]), float(case["rows"])
    total = rows
    if kind == "hetero":
        total = rows + (case["islands"] - 1) * (rows - case["rmin"]) / math.log(rows / case["rmin"])
    cell = 8.0 * 4.0 * total + cands * case.get("islands", 1) * 512.0
    if kind == "order":
        return {"bytes": cell, "flops": float(cands * case["trials"] * rows * (value + 3.0))}
    passes = 4.0 if case["iters"] else 1.0
    return {"bytes": cell, "flops": float(cands * total * passes * (3.0 * value + 2.0 * k + 6.0))}


def tolerance(case):
    """About four times what was measured against exact(), or where that has no
    value, with the rows summed in tiles of another size and against the plain
    64-bit arm."""
    kind = case["kind"]
    if kind in ("eval", "score"):  # f32 programs, f64 sums: 6e-8
        return {"rel": 4e-7, "max": 2e-5}
    if kind == "pool":  # the programs are whole numbers; the losses f32 programs
        return {"rel": 4e-7, "max": 2e-5}
    if kind == "hetero" or case.get("metric") == 4:
        # IRLS stopped after its rounds is no optimum: f32 and f64 rows leave
        # it 0.1 apart in the constants and 4e-3 in the loss.
        return {"rel": 2e-2, "max": 0.9, "differ": 0.01}
    if kind == "fit":  # 2e-5 in the constants of the slowest to converge
        return {"rel": 1e-4, "max": 1e-3, "differ": 0.01}
    if kind == "corr":
        return {"rel": 1e-5, "max": 1e-3, "differ": 0.01}
    if kind == "implicit":  # the difference Jacobian's noise: 3e-10
        return {"rel": 1e-8, "max": 1e-6, "differ": 0.01}
    return {"rel": 1e-12, "max": 1e-10}  # f64 rows, exact statistics: 0


# ---- the same in 64 bits ------------------------------------------------------------

DEV = "cuda" if torch.cuda.is_available() else "cpu"


def _value(t, x, c):
    """A tuple program over the f64 rows x with constants c."""
    if t[0] == "c":
        return c[t[1]]
    if t[0] == "k":
        return torch.tensor(t[1], dtype=torch.float64, device=x.device)
    if t[0] == "x":
        return x[t[1]]
    k = [_value(u, x, c) for u in t[1:]]
    return {"+": torch.add, "-": torch.sub, "*": torch.mul, "/": torch.div, "sin": torch.sin,
            "cos": torch.cos, "exp": torch.exp, "log": torch.log, "tanh": torch.tanh,
            "square": torch.square}[t[0]](*k)


def _derivatives(t, x, c, want):
    """Value and derivatives by the constants ("c") or the inputs ("x"), as a
    dict of slot or column to tensor."""
    if t[0] in ("c", "x", "k"):
        one = {t[1]: torch.ones((), dtype=torch.float64, device=x.device)}
        return _value(t, x, c), (one if t[0] == want else {})
    kids = [_derivatives(u, x, c, want) for u in t[1:]]
    v = [k[0] for k in kids]
    if t[0] in ("+", "-", "*", "/"):
        a, b = v
        r = _value((t[0], ("c", 0), ("c", 1)), x, v)
        part = {"+": (1.0, 1.0), "-": (1.0, -1.0), "*": (b, a), "/": (1.0 / b, -r / b)}[t[0]]
    else:
        a = v[0]
        r = _value((t[0], ("c", 0)), x, v)
        part = ({"sin": torch.cos, "cos": lambda u: -torch.sin(u), "exp": lambda u: r,
                 "log": lambda u: 1.0 / u, "tanh": lambda u: 1.0 - r * r,
                 "square": lambda u: 2.0 * u}[t[0]](a),)
    out = {}
    for (_, g), p in zip(kids, part):
        for j, h in g.items():
            out[j] = out[j] + p * h if j in out else p * h
    return r, out


def _descend(residual, c, steps=60):
    """Damped Gauss-Newton to the least-squares optimum; residual(c, True)
    gives the residual and its Jacobian."""
    lam, (r, J) = 1e-3, residual(c, True)
    best = float(r @ r)
    for _ in range(steps):
        H, g = J.T @ J, J.T @ r
        while True:
            D = torch.diag(torch.diagonal(H) * lam)
            trial = c - torch.linalg.solve(H + D, g)
            q = residual(trial, False)
            loss = float(q @ q)
            if loss <= best or lam > 1e8:
                break
            lam *= 8.0
        if not loss <= best:
            break
        done = float((trial - c).abs().max()) < 1e-13 * (1.0 + float(c.abs().max()))
        c, best, lam = trial, loss, max(lam / 10.0, 1e-12)
        if done:
            break
        r, J = residual(c, True)
    return c, best


def _fit_exact(cands, x, y):
    n = x.shape[1]
    out = []
    for t, c0 in cands:
        def residual(c, jac):
            if not jac:
                return (_value(t, x, c) - y).expand(n)
            f, g = _derivatives(t, x, c, "c")
            J = torch.stack([g[j].expand(n) for j in range(len(c0))], 1)
            return (f - y).expand(n), J
        out.append(_descend(residual, torch.tensor(c0, dtype=torch.float64, device=DEV)))
    return out


def _distance(t, x, c):
    f, g = _derivatives(t, x, c, "x")
    return f / torch.sqrt(sum(v * v for v in g.values()))


def exact(case, seed):
    kind = case["kind"]
    if kind == "pool":
        return None
    # Fits cost some thirty assemblies a candidate here; the largest are left out.
    if kind in ("fit", "hetero", "corr", "implicit"):
        cost = case["rows"] * case["candidates"] * (case["kmin"] + case["kmax"])
        if kind == "hetero" or case.get("metric") or cost > 4e8 or case["candidates"] > 250:
            return None
    d = _inputs(case, seed)
    x = torch.tensor(np.asarray(d["x"], np.float64), device=DEV)
    y = torch.tensor(np.asarray(d["y"], np.float64), device=DEV)
    n = case["rows"]
    if kind == "eval":
        out = []
        for t in d["trees"]:
            r = (_value(t, x, ()) - y).expand(n)
            row = {0: lambda: r * r, 1: lambda: torch.log1p(r * r), 4: r.abs}[case["loss"]]()
            out.append(row.sum())
        return {"loss": torch.stack(out)}
    if kind == "score":
        out = [_score(_value(t, x, ()).expand(n), y, case["score"]) for t in d["trees"]]
        return {"score": torch.stack(out), "status": None}
    if kind == "fit":
        got = _fit_exact(d["cands"], x, y)
        return {"c": torch.cat([c for c, _ in got]), "loss": torch.tensor([v for _, v in got],
                                                                       dtype=torch.float64),
                "status": None}
    if kind == "corr":
        cs, loss = [], []
        for (t, _), (c, best) in zip(d["cands"], _fit_exact(d["cands"], x, y)):
            rho = math.sqrt(max(0.0, 1.0 - best / float(((y - y.mean()) ** 2).sum())))
            c = c.clone()
            c[0], c[-1] = torch.sign(c[0]), 0.0
            cs.append(c)
            loss.append(1.0 - rho)
        return {"c": torch.cat(cs), "loss": torch.tensor(loss, dtype=torch.float64),
                "status": None}
    if kind == "implicit":
        if not case["iters"]:
            out = [_distance(t, x, torch.tensor(c, dtype=torch.float64, device=DEV)).abs().mean()
                   for t, c in d["cands"]]
            return {"score": torch.stack(out), "status": None}
        cs, loss = [], []
        for t, c0 in d["cands"]:
            def residual(c, jac):
                r = _distance(t, x, c)
                if not jac:
                    return r
                cols = []
                for j in range(len(c)):
                    h = torch.zeros_like(c)
                    h[j] = 1e-5
                    cols.append((_distance(t, x, c + h) - _distance(t, x, c - h)) / 2e-5)
                return r, torch.stack(cols, 1)
            c, best = _descend(residual, torch.tensor(c0, dtype=torch.float64, device=DEV), 15)
            cs.append(c)
            loss.append(best)
        return {"c": torch.cat(cs), "loss": torch.tensor(loss, dtype=torch.float64),
                "status": None}
    return _order_exact(case, d, x, y)


def _score(p, y, kind):
    if not bool(torch.isfinite(p).all()) or bool((p.abs() > 1e30).any()):
        return torch.tensor(math.inf, dtype=torch.float64, device=p.device)
    r = p - y
    if kind == 5:
        a, b = p - p.mean(), y - y.mean()
        ss = (a * a).sum()
        if not float(ss) > 0.0:
            return torch.ones((), dtype=torch.float64, device=p.device)
        return 1.0 - ((a * b).sum() / (ss.sqrt() * (b * b).sum().sqrt())).abs()
    return {0: lambda: (r * r).mean(), 1: lambda: r.abs().mean(),
            2: lambda: torch.log1p(r * r).mean(), 4: lambda: r.abs().max()}[kind]()


def _ranks(v):
    """Doubled centred average ranks."""
    u, inv, cnt = torch.unique(v, return_inverse=True, return_counts=True)
    end = torch.cumsum(cnt, 0)
    return ((end - cnt) + end - len(v))[inv].to(torch.float64)


def _order_exact(case, d, x, y):
    n, what = case["rows"], case["what"]
    res = {"value": [], "sums": [], "max": [], "lo": [], "hi": []}
    B = _ranks(y) if what == "ranks" else None
    for s in range(len(d["c"])):
        t, c0 = d["cands"][s // case["trials"]]
        c = torch.tensor(d["c"][s, :len(c0)], dtype=torch.float64, device=DEV)
        p = _value(t, x, c).expand(n)
        r = (p - y).abs()
        if what == "median":
            v = torch.sort(r).values
            res["value"].append(v[n // 2] if n % 2 else 0.5 * (v[n // 2 - 1] + v[n // 2]))
        elif what == "quartiles":
            v = torch.sort(r).values
            res["value"].append(v[n // 4:max(3 * n // 4, n // 4 + 1)].mean())
        elif what == "ranks":
            A = _ranks(p)
            res["sums"].append(torch.stack([(A * B).sum(), (A * A).sum()]))
        else:
            res["max"].append(r.max())
            if what == "level":
                b = _derivatives(t, x, c, "c")[1][0].expand(n)
                q = p - y
                ends = torch.stack([(-LEVEL - q) / b, (LEVEL - q) / b])
                lo, hi = ends.min(0).values[b != 0].max(), ends.max(0).values[b != 0].min()
                veto = bool(((b == 0) & (q.abs() > LEVEL)).any())
                res["lo"].append(torch.full_like(lo, math.inf) if veto else lo)
                res["hi"].append(torch.full_like(hi, -math.inf) if veto else hi)
    if what in ("median", "quartiles"):
        return {"value": torch.stack(res["value"]), "status": None}
    if what == "ranks":
        return {"sums": torch.stack(res["sums"]), "target": float((B * B).sum()), "status": None}
    out = {"max": torch.stack(res["max"]), "row": None}
    if what == "level":
        out["lo"], out["hi"] = torch.stack(res["lo"]), torch.stack(res["hi"])
    return out
