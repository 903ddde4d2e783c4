"""Fits whose gradient tape does not fit the U register file: the 4-row
assembly kernels then keep part of it in B (VMC_TAPE_B) or in LDS
(VMC_TAPE_L).  Sums of k terms c * basis(x) need one tape value per term, so
k walks over the edges of the three forms (15 U slots less the inputs, 8 B
slots), with a row count that ends inside a 256-row step."""
import ctypes as C

import numpy as np
import pytest

import oracle
from rcsr_hip import host, lib
from rcsr_hip.expr import (ADD, COS, COSH, CUBE, ERF, EXP, GAUSS, MUL, SIG, SIN, SQUARE, TANH,
                           const, node, var)

INPUTS_IN_U, TAPE_B, SMALL_B, TAPE_L = 1, 8, 16, 32


UNARY = [SIN, SQUARE, COS, TANH, EXP, CUBE, GAUSS, SIG, ERF, COSH]


def _basis(i, nv):
    return node(UNARY[(i // nv) % len(UNARY)], var(i % nv))


def _tree(k, nv, inner):
    """k constants: `inner` terms c * exp(c' * x^2), the others c * basis."""
    terms = [node(MUL, const(0.6), node(EXP, node(MUL, const(-0.3 - 0.1 * i),
                                                  node(SQUARE, var(i % nv)))))
             for i in range(inner)]
    terms += [node(MUL, const(0.1 * (i + 1)), _basis(i, nv)) for i in range(k - 2 * inner)]
    t = terms[0]
    for u in terms[1:]:
        t = node(ADD, t, u)
    return t


def _compiled(plan, nv, flags):
    L = lib.load()
    L.rch_fitvm_compile.restype = C.c_int
    w = np.ascontiguousarray(plan.words)
    f, r, info = np.zeros(1024, np.uint32), np.zeros(2048, np.uint32), np.zeros(6, np.int32)
    rc = L.rch_fitvm_compile(lib.ptr(w, lib.u32p), len(w), plan.nconst, nv, 258 * 4, flags,
                             lib.ptr(f, lib.u32p), 1024, lib.ptr(r, lib.u32p), 2048,
                             lib.ptr(info, lib.i32p))
    return rc, info


CASES = [(12, 3, 0), (13, 3, 0), (14, 3, 1), (15, 4, 0), (16, 2, 0), (18, 3, 0), (20, 3, 2),
         (19, 3, 0), (18, 7, 0), (20, 5, 2), (10, 1, 1)]


def test_the_cases_reach_every_form():
    forms = set()
    for k, nv, inner in CASES:
        plan = host.gpu_fit_plan(_tree(k, nv, inner))
        u = _compiled(plan, nv, INPUTS_IN_U)[0]
        rb, ib = _compiled(plan, nv, INPUTS_IN_U | SMALL_B | TAPE_B)
        rl, il = _compiled(plan, nv, INPUTS_IN_U | SMALL_B | TAPE_L)
        assert rl == 0 and il[5] <= 16 and (rb != 0 or ib[3] <= 8)
        forms.add("U" if u == 0 else "B" if rb == 0 else "L")
    assert forms == {"U", "B", "L"}


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [777, 20001])
@pytest.mark.parametrize("k,nv,inner", CASES)
def test_fits_of_every_tape_form_match_the_other_kernels(k, nv, inner, rows):
    rng = np.random.default_rng(k * 100 + nv)
    x = rng.uniform(-2.0, 2.0, size=(rows, nv))
    tree = _tree(k, nv, inner)
    truth = oracle.predict(tree.with_constants(list(rng.uniform(-1.0, -0.2, k))), x)
    y = truth + 0.1 * rng.standard_normal(rows)
    ev = host.GpuEvaluator(np.ascontiguousarray(x.T, np.float32).reshape(-1), rows, nv,
                           y.astype(np.float32))
    assert ev.set_fit_data(np.ascontiguousarray(x.T).reshape(-1), y)
    print(f"tape fit k={k} nv={nv} inner={inner} rows={rows}", flush=True)
    (out,), ms = ev.fit_batch([host.gpu_fit_plan(tree)], 30, 0)
    assert ms >= 0 and host.fit_status_usable(out.status)
    # The reported loss is the exact one of the returned constants, or that of
    # the f32 rows (2^-24 a value, a few of them a row) where a solve failed
    # (status 5: the most collinear of these sums).
    tol = 1e-6 if out.status == 5 else 1e-11
    assert abs(oracle.sse(tree.with_constants(out.c), x, y) - out.sse) <= tol * out.sse
    # With 2 rows per lane these programs run on the 2-row or the general
    # kernel: the same f32 arithmetic per node and the same row order in the
    # Gram sums, so the fit's steps are the same ones.
    ev.set_tuning(host.TUNE_FIT_ROWS_PER_LANE, 2)
    (ref,), ms = ev.fit_batch([host.gpu_fit_plan(tree)], 30, 0)
    assert ms >= 0 and ref.status == out.status
    assert abs(ref.sse - out.sse) <= 1e-12 * ref.sse
    ev.close()
