/*
 * The implicit arm's four-wide sweep on gfx950: im_pass_kernel's contract
 * (rc_implicit.hip) for programs without guarded operators, with at most
 * IM_WDEPTH values below the top of their evaluation stack, over at most IM_WNV
 * input columns.  Without LOG, SQRT, TAN and POW the guarded value of
 * expr::eval is the value itself, so a stack entry is the value and the input
 * tangents, and a stack of four entries fits one 16-element vector.
 *
 * A wave is an interpreter of wave-uniform records, bound by the latency of
 * its dispatch and of dependent f64 arithmetic; four sweeps side by side share
 * the dispatch and fill the waits: four of the 2k + 1 distances of a row in the
 * Jacobian pass, four rows in the others.  Every operation is the one that
 * im_fast_kernel does, in its order.  128 candidates of 2 to 7 constants x
 * 65 537 rows: 97 ms a fit with im_fast_kernel, 39 with this one (a Jacobian
 * pass 4.4 ms, a residual pass 0.33).  This file is
 * built with uniform regions left unstructured.
 */
#include "rc_implicit_dev.h"

namespace {

__device__ __forceinline__ unsigned im_uniform(unsigned op)
{
    return (unsigned)__builtin_amdgcn_readfirstlane((int)op);
}

/* Four values and local partials of a unary operator (im_unary_all's). */
struct ImFour {
    double v[4], p[4];
};
__device__ __noinline__ ImFour im_unary4(uint32_t op_, double a0, double a1, double a2, double a3)
{
    const uint32_t op = im_uniform(op_);
    const double x[4] = {a0, a1, a2, a3};
    ImFour u;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const double a = x[w];
        if (op == OP_SIN || op == OP_COS) {
            /* One argument reduction for both: sincos's outputs are sin's and
               cos's bits on gfx950 (128 fits x 65 537 rows 39.9 ->
               37.9 ms). */
            double sn, cs;
            sincos(a, &sn, &cs);
            u.v[w] = op == OP_SIN ? sn : cs;
            u.p[w] = op == OP_SIN ? cs : -sn;
            continue;
        }
        const double v = im_value(op, a, 0.0);
        double p;
        switch (op) {
            case OP_EXP: p = a > 700.0 ? exp(a) : v; break;
            case OP_ABS: p = a >= 0.0 ? 1.0 : -1.0; break;
            case OP_SINH: p = cosh(a); break;
            case OP_COSH: p = sinh(a); break;
            case OP_TANH: p = 1.0 - v * v; break;
            case OP_SIG: p = v * (1.0 - v); break;
            case OP_GAUSS: p = (-2.0 * a) * v; break;
            case OP_CUBE: p = 3.0 * a * a; break;
            case OP_ERF: p = 2.0 * IM_INV_SQRT_PI * exp(-a * a); break;
            case OP_ERFC: p = -2.0 * IM_INV_SQRT_PI * exp(-a * a); break;
            default: p = 0.0; break;
        }
        u.v[w] = v;
        u.p[w] = p;
    }
    return u;
}

/* Four sweeps: evaluation w at the inputs x[w] and the constants c, slot pj[w]
   replaced by cpj[w].  out[w] is the signed distance (metric 0) or f (metric
   1), ok[w] whether the row is defined. */
template <int NV>
__device__ __forceinline__ void im_wide_distance(const uint32_t *__restrict__ r4, int m,
                                                 const double *__restrict__ c, const int (&pj)[4],
                                                 const double (&cpj)[4], const double (&x)[4][NV],
                                                 int metric, double (&out)[4], bool (&ok)[4])
{
    /* Entry e of evaluation w: the value in element e of S_w, the tangents in
       e + 4, e + 8, e + 12 (one indexed move each). */
    im_d16 S0, S1, S2, S3;
    double v[4] = {0.0, 0.0, 0.0, 0.0}, t[4][NV];
#pragma unroll
    for (int w = 0; w < 4; ++w)
#pragma unroll
        for (int q = 0; q < NV; ++q) t[w][q] = 0.0;
    int sp = -1; /* entries below the top; -1: empty */
    auto push = [&](im_d16 &S, int w) {
        S[sp] = v[w];
#pragma unroll
        for (int q = 0; q < NV; ++q) S[sp + 4 * (q + 1)] = t[w][q];
    };
    for (int i = 0; i < m; ++i) {
        const uint32_t op = r4[4 * i], slot = r4[4 * i + 3];
        if (op == OP_CONST || op == OP_VAR) {
            if (sp >= 0) {
                push(S0, 0);
                push(S1, 1);
                push(S2, 2);
                push(S3, 3);
            }
            ++sp;
            if (op == OP_CONST) {
                const double cv = c[slot];
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    v[w] = (int)slot == pj[w] ? cpj[w] : cv;
#pragma unroll
                    for (int q = 0; q < NV; ++q) t[w][q] = 0.0;
                }
            } else {
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    v[w] = x[w][0];
#pragma unroll
                    for (int q = 1; q < NV; ++q) v[w] = (int)slot == q ? x[w][q] : v[w];
#pragma unroll
                    for (int q = 0; q < NV; ++q) t[w][q] = (int)slot == q ? 1.0 : 0.0;
                }
            }
        } else if (im_is_bin(op)) {
            --sp;
            auto combine = [&](const im_d16 &S, int w) {
                const double va = S[sp], vb = v[w];
                double ta[NV];
#pragma unroll
                for (int q = 0; q < NV; ++q) ta[q] = S[sp + 4 * (q + 1)];
                if (op == OP_ADD) {
                    v[w] = va + vb;
#pragma unroll
                    for (int q = 0; q < NV; ++q) t[w][q] = ta[q] + t[w][q];
                } else if (op == OP_SUB) {
                    v[w] = va - vb;
#pragma unroll
                    for (int q = 0; q < NV; ++q) t[w][q] = ta[q] - t[w][q];
                } else if (op == OP_MUL) {
                    v[w] = va * vb;
#pragma unroll
                    for (int q = 0; q < NV; ++q) t[w][q] = im_lm(vb, ta[q]) + im_lm(va, t[w][q]);
                } else { /* DIV */
                    v[w] = fabs(vb) < 1e-12 ? RC_F64_NAN : va / vb;
#pragma unroll
                    for (int q = 0; q < NV; ++q) {
                        const double b_ = t[w][q];
                        t[w][q] = im_ld(ta[q], vb) + (b_ == 0.0 ? 0.0 : -(va * b_) / (vb * vb));
                    }
                }
            };
            combine(S0, 0);
            combine(S1, 1);
            combine(S2, 2);
            combine(S3, 3);
        } else if (op == OP_SQUARE || op == OP_NEG) {
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const double p = op == OP_SQUARE ? 2.0 * v[w] : -1.0;
#pragma unroll
                for (int q = 0; q < NV; ++q) t[w][q] = im_lm(p, t[w][q]);
                v[w] = op == OP_SQUARE ? v[w] * v[w] : -v[w];
            }
        } else {
            const ImFour u = im_unary4(op, v[0], v[1], v[2], v[3]);
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                v[w] = u.v[w];
#pragma unroll
                for (int q = 0; q < NV; ++q) t[w][q] = im_lm(u.p[w], t[w][q]);
            }
        }
    }
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        bool good = isfinite(v[w]);
        out[w] = v[w];
        if (metric == 0) {
            double norm_sq = 0.0;
#pragma unroll
            for (int q = 0; q < NV; ++q) {
                good = good && isfinite(t[w][q]);
                norm_sq += t[w][q] * t[w][q];
            }
            const double norm = sqrt(norm_sq);
            out[w] = v[w] / norm;
            good = good && isfinite(norm) && norm > 0.0 && isfinite(out[w]);
        }
        ok[w] = good;
    }
}

template <int MODE, int NV>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void im_wide_kernel(
    const ImItem *__restrict__ items, int nitems, const ImCand *__restrict__ cands,
    const uint32_t *__restrict__ rec, const double *__restrict__ cs, int kmax,
    const double *__restrict__ cols64, const double *__restrict__ w64, int n, int metric,
    double *__restrict__ part, int pstride, int *__restrict__ bad, const int *__restrict__ run)
{
    constexpr int ROWS = MODE == IM_JAC ? 64 : 256; /* of a step */
    const int it_i = blockIdx.x;
    if (it_i >= nitems) return;
    const ImItem it = items[it_i];
    if (run && !run[it.cand]) return;
    const ImCand d = cands[it.cand];
    if (d.fast != 2) return;
    const int lane = threadIdx.x;
    const uint32_t *r4 = rec + d.off;
    const double *c = cs + (size_t)it.cand * (size_t)kmax;
    const int k = d.k, K1 = k + 1; /* [J | r] columns */
    __shared__ double J[MODE == IM_JAC ? 64 : 1][IM_KMAX + 2];
    im_d4 acc00 = {0.0, 0.0, 0.0, 0.0}, acc10 = acc00, acc11 = acc00;
    if (MODE == IM_JAC) {
        for (int q = lane; q < 64 * (IM_KMAX + 2); q += 64) (&J[0][0])[q] = 0.0;
        __syncthreads();
    }
    double s0 = 0.0, s1 = 0.0;
    int flag = 0;
    const int row_end = it.row0 + it.rows;
    double *p = part + (size_t)it_i * (size_t)pstride;
    double t0 = 0.0, t1 = 0.0;
    int sub_end = it.row0 + d.sub;
    for (int base = it.row0; base < row_end; base += ROWS) {
        double x[4][NV], wt[4];
        bool use[4];
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            if (MODE == IM_JAC && w > 0) {
                wt[w] = wt[0];
                use[w] = use[0];
#pragma unroll
                for (int q = 0; q < NV; ++q) x[w][q] = x[0][q];
                continue;
            }
            const int row = base + 64 * w + lane;
            const bool live = row < row_end;
            const int rr = live ? row : it.row0;
            wt[w] = w64 ? w64[rr] : 1.0;
            const bool fine = isfinite(wt[w]) && wt[w] >= 0.0;
            if (live && !fine) flag |= 2;
            use[w] = live && fine && wt[w] > 0.0;
#pragma unroll
            for (int q = 0; q < NV; ++q) x[w][q] = cols64[(size_t)q * (size_t)n + (size_t)rr];
        }
        double out[4];
        bool ok[4];
        if (MODE != IM_JAC) {
            const int none[4] = {-1, -1, -1, -1};
            const double zero[4] = {0.0, 0.0, 0.0, 0.0};
            im_wide_distance<NV>(r4, d.m, c, none, zero, x, MODE == IM_SCORE ? metric : 0, out, ok);
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                if (!use[w]) continue;
                if (!ok[w]) {
                    flag |= 1;
                } else if (MODE == IM_SCORE) {
                    s0 += wt[w] * fabs(out[w]);
                    s1 += wt[w];
                } else {
                    const double r = sqrt(wt[w]) * out[w];
                    s0 += r * r;
                }
            }
        } else {
            /* Positions 2 j and 2 j + 1 are c_j + h and c_j - h, position 2 k
               the distance at c; the last sweep repeats it where it has room. */
            const double sw = use[0] ? sqrt(wt[0]) : 0.0;
            for (int e = 0; e <= 2 * k; e += 4) {
                int pj[4];
                double cp[4], h[2];
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const int j = (e + w) >> 1;
                    pj[w] = j < k ? j : -1;
                    const double cj = j < k ? c[j] : 0.0;
                    const double hw = 1e-6 * (1.0 + fabs(cj));
                    cp[w] = (w & 1) ? cj - hw : cj + hw;
                    if (!(w & 1)) h[w >> 1] = hw;
                }
                im_wide_distance<NV>(r4, d.m, c, pj, cp, x, 0, out, ok);
                bool good = true;
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int j = (e >> 1) + u;
                    good = good && ok[2 * u] && ok[2 * u + 1];
                    if (j < k) {
                        const double g = (sw * out[2 * u] - sw * out[2 * u + 1]) / (2.0 * h[u]);
                        good = good && isfinite(g);
                        J[lane][j] = use[0] ? g : 0.0;
                    } else if (j == k) {
                        const double r = sw * out[2 * u];
                        good = good && isfinite(r);
                        J[lane][k] = use[0] ? r : 0.0;
                    }
                }
                if (use[0] && !good) flag |= 1;
            }
            __syncthreads();
            {
                /* Operand of lane (col, sub) for rows 4 t + sub: A and B of
                   the MFMA are the same block of J. */
                const int col = lane & 15, sub = lane >> 4;
                const int col1 = (16 + col < IM_KMAX + 2) ? 16 + col : IM_KMAX + 1;
#pragma unroll 4
                for (int t4 = 0; t4 < 16; ++t4) {
                    const double a0 = J[4 * t4 + sub][col];
                    acc00 = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, a0, acc00, 0, 0, 0);
                    if (K1 > 16) {
                        const double a1 = J[4 * t4 + sub][col1];
                        acc10 = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, a0, acc10, 0, 0, 0);
                        acc11 = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, a1, acc11, 0, 0, 0);
                    }
                }
            }
            __syncthreads();
        }
        /* The end of a sub-tile: its sums go onto the item's (as in
           im_fast_kernel). */
        if (base + ROWS >= sub_end || base + ROWS >= row_end) {
            const bool add = sub_end != it.row0 + d.sub;
            /* rc_here: 640 Jacobian fits x 131 072 rows of two inputs 114.4 ->
               112.8 ms; three inputs keep 112 bytes of scratch less but take
               133.2 ms for 130.4. */
            const int at = NV < 3 ? rc_here(lane) : lane;
            if (MODE == IM_JAC) {
                const int jj = at & 15;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int ii = (at >> 4) + 4 * r, i1 = 16 + ii;
                    if (ii >= jj && ii < K1) rc_put(p + ii * (ii + 1) / 2 + jj, acc00[r], add);
                    if (i1 < K1) rc_put(p + i1 * (i1 + 1) / 2 + jj, acc10[r], add);
                    if (ii >= jj && i1 < K1) rc_put(p + i1 * (i1 + 1) / 2 + 16 + jj, acc11[r], add);
                    acc00[r] = acc10[r] = acc11[r] = 0.0;
                }
            } else {
                t0 = rc_scalar(t0 + rc_wave_sum_f64(s0));
                t1 = rc_scalar(t1 + rc_wave_sum_f64(s1));
                s0 = s1 = 0.0;
            }
            sub_end += d.sub;
        }
    }
    int f = flag;
    for (int off = 32; off > 0; off >>= 1) f |= __shfl_xor(f, off, 64);
    if (MODE != IM_JAC && lane == 0) {
        p[0] = t0;
        p[1] = t1;
    }
    if (lane == 0) bad[it_i] = f;
}

template <int MODE>
void launch_mode(int nv, int ni, hipStream_t s, const ImItem *items, const ImCand *cands,
                 const uint32_t *rec, const double *cs, int kmax, const double *cols64,
                 const double *w64, int n, int metric, double *part, int pstride, int *bad,
                 const int *run)
{
#define IM_WIDE(NV)                                                                                \
    im_wide_kernel<MODE, NV><<<ni, 64, 0, s>>>(items, ni, cands, rec, cs, kmax, cols64, w64, n, \
                                              metric, part, pstride, bad, run)
    if (nv == 1) IM_WIDE(1);
    else if (nv == 2) IM_WIDE(2);
    else IM_WIDE(3);
#undef IM_WIDE
}

} /* namespace */

void im_launch_wide(int mode, int nv, int ni, hipStream_t s, const ImItem *items,
                    const ImCand *cands, const uint32_t *rec, const double *cs, int kmax,
                    const double *cols64, const double *w64, int n, int metric, double *part,
                    int pstride, int *bad, const int *run)
{
    if (ni <= 0) return;
    if (mode == IM_SCORE)
        launch_mode<IM_SCORE>(nv, ni, s, items, cands, rec, cs, kmax, cols64, w64, n, metric, part,
                              pstride, bad, run);
    else if (mode == IM_RSS)
        launch_mode<IM_RSS>(nv, ni, s, items, cands, rec, cs, kmax, cols64, w64, n, metric, part,
                            pstride, bad, run);
    else
        launch_mode<IM_JAC>(nv, ni, s, items, cands, rec, cs, kmax, cols64, w64, n, metric, part,
                            pstride, bad, run);
}
