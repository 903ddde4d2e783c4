/*
 * Row kernels of the order and maximum stages on gfx950: sort keys and tile
 * maxima of candidate predictions in f64 (reference eval.cu:2952-2982,
 * 4383-4419, 4505-4600).  They are single-wave interpreters of wave-uniform
 * words with their operands in registers, where the general kernels of
 * rc_order.hip keep every node's value in per-lane scratch, and they run one
 * wave per (segment, row tile).  Built with uniform regions left unstructured
 * and without contraction, so every product and sum is rounded on its own.
 *
 * 256 segments (64 candidates x 4 constant vectors), value in ms before ->
 * after: keys over 262 144 rows 14.9 -> 1.1; maximum with a level over
 * 100 003 rows 35.0 -> 1.2.  Both are bound by the f64 arithmetic of the
 * operators and the dispatch around it; the keys are 0.54 GB of writes, 0.1 ms.
 */
#include "rc_fit_dev.h"
#include "rc_fitvm_dev.h"
#include "rc_order_kern.h"

#include <math.h>

namespace {

constexpr unsigned long long OR_BAD = 0xFFFFFFFFFFFFFFFFull;

/* Order-preserving 64-bit key of a finite f64 (-0.0 keyed as +0.0). */
__device__ __forceinline__ unsigned long long or_rank_key(double v)
{
    if (v == 0.0) v = 0.0;
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}

__device__ __forceinline__ bool or_bad_row(double pred, double r)
{
    return !isfinite(pred) || fabs(pred) > 1e30 || !isfinite(r);
}

/* Predictions of the rows q[0..3] on a set's value stream. */
__device__ __forceinline__ vm_d4 or_value(const uint2 *code, int words, const double *cst,
                                          const OrRows &R, const int (&q)[4])
{
    typedef VmPack<vm_d4> P;
    dv8 U0 = (dv8)(0.0), U1 = U0, U2 = U0, U3 = U0, B = U0;
#pragma unroll
    for (int v = 0; v < VM_MAX_VARS; ++v)
        if (v < R.v) {
            const double *col = R.cols64 + (size_t)v * (size_t)R.n;
            P::set(U0, U1, U2, U3, v, (vm_d4){col[q[0]], col[q[1]], col[q[2]], col[q[3]]});
        }
    return vm_forward<vm_d4, false>(code, words, cst, U0, U1, U2, U3, U0, U1, U2, U3, B, B, B, B);
}

template <bool RANK>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3))) void or_keys_kernel(
    const int *__restrict__ segs, const OrSet *__restrict__ sets, const uint32_t *__restrict__ code,
    const double *__restrict__ c0, int kmax, int ntrials, OrRows R, int tiles, int tile_rows,
    unsigned long long *__restrict__ keys, uint32_t *__restrict__ row_of, int *__restrict__ status)
{
    const int li = blockIdx.x / tiles, tile = blockIdx.x - li * tiles;
    const int seg = segs[li];
    const OrSet d = sets[seg / ntrials];
    const double *cst = c0 + (size_t)seg * (size_t)kmax;
    const int lane = threadIdx.x;
    const int begin = tile * tile_rows, end = min(R.n, begin + tile_rows);
    unsigned long long *k = keys + (size_t)seg * (size_t)R.n;
    int bad = 0;
    for (int base = begin; base < end; base += 256) {
        int q[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) q[r] = min(base + 64 * r + lane, R.n - 1);
        const vm_d4 pred = or_value((const uint2 *)(code + d.t_off), d.t_m, cst, R, q);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = base + 64 * r + lane;
            if (row >= end) continue;
            unsigned long long key;
            if (RANK) {
                key = isfinite(pred[r]) ? or_rank_key(pred[r]) : OR_BAD;
                row_of[(size_t)seg * (size_t)R.n + (size_t)row] = (uint32_t)row;
            } else {
                const double rr = pred[r] - R.y64[row];
                key = or_bad_row(pred[r], rr) ? OR_BAD
                                              : (unsigned long long)__double_as_longlong(fabs(rr));
            }
            bad |= key == OR_BAD;
            k[row] = key;
        }
    }
    if (bad) status[seg] = 2;
}

/* Prediction and its derivative by constant slot j for two rows a lane, in one
   forward sweep over the post-order records: a value and a tangent per stack
   entry, the top in fixed registers, the entries below in a 16-element vector
   a row (values in 0..7, tangents in 8..15) indexed by the wave-uniform depth.
   The local partials are ft_rec_hand_down's.

   The constant is one leaf, so its derivative is the product of the partials on
   one path, which the adjoint sweep takes from the root down and this one from
   the leaf up.  The sweep from the root ends at the first partial of zero (the
   derivative is zero, whatever is below it) or that is not finite (neither is
   the derivative).  Seen from the leaf that is the last such partial: it is
   noted, in place of one noted before, and the product starts again from 1
   above it.  The adjoint of a node above that is the last of these products
   over the node's own, so the least and the greatest binary exponent of the
   products say whether any adjoint left 2^+-800; while none did, and no product
   leaves 2^+-1000, both sweeps stay in the normal range at every step and agree
   to rounding.  Any other row, and one that ends in a partial that is not
   finite, sends its segment to the general kernel. */
enum { OR_ZERO = 1, OR_WILD = 4, OR_REDO = 16 }; /* the first two shifted by the row */
constexpr double OR_BIG = 0x1p1000, OR_SMALL = 0x1p-1000;
constexpr int OR_ADJOINT = 800;
/* A factor that an adjoint meets before another one. */
constexpr double OR_FACTOR_BIG = 0x1p200, OR_FACTOR_SMALL = 0x1p-200;

/* A node's values and tangents and what its partials were (OR_*). */
struct OrDual {
    double v[2], t[2];
    int ev;
};

__device__ __forceinline__ bool or_in_range(double u)
{
    return fabs(u) >= OR_SMALL && fabs(u) <= OR_BIG;
}
__device__ __forceinline__ bool or_mild(double f)
{
    return fabs(f) >= OR_FACTOR_SMALL && fabs(f) <= OR_FACTOR_BIG;
}
/* The tangent t through the partial p; off the path both stay zero. */
__device__ __forceinline__ double or_tan(double p, double t, int r, int &ev)
{
    if (t == 0.0) return 0.0;
    if (p == 0.0 || !isfinite(p)) {
        ev |= (p == 0.0 ? OR_ZERO : OR_WILD) << r;
        return 1.0;
    }
    const double u = p * t;
    if (!or_in_range(u)) ev |= OR_REDO;
    return u;
}

__device__ __noinline__ OrDual or_unary(unsigned op_, double v0, double v1, double t0, double t1)
{
    const unsigned op = vm_uniform(op_);
    const double v[2] = {v0, v1}, t[2] = {t0, t1};
    OrDual o;
    o.ev = 0;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        o.v[r] = ft_unary(op, v[r]);
        o.t[r] = t[r] == 0.0
                     ? 0.0
                     : or_tan(ft_unary_partial<double>(op, v[r], o.v[r]), t[r], r, o.ev);
    }
    return o;
}

/* A division or a power with the path's tangent t on its left or right side:
   t / d and -t l / (d d), t d pow(l, d - 1) and t pow(l, d) log(l) for l > 0,
   else 0.  In the last three an adjoint meets the factors f and g one by one. */
__device__ __noinline__ OrDual or_divide_or_pow(unsigned op_, double l0, double l1, double d0,
                                                double d1, double t0, double t1, int left)
{
    const unsigned op = vm_uniform(op_);
    const double lv[2] = {l0, l1}, dv[2] = {d0, d1}, tv[2] = {t0, t1};
    OrDual o;
    o.ev = 0;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const double l = lv[r], d = dv[r], t = tv[r];
        o.v[r] = ft_binary(op, l, d);
        o.t[r] = 0.0;
        if (t == 0.0) continue;
        double u = 0.0, f = 1.0, g = 0.0;
        bool mild = true;
        if (op == OP_DIV) {
            const double q = left ? d : d * d;
            if (!left) f = l;
            g = isinf(q) ? 0.0 : q == 0.0 ? RC_F64_NAN : q;
            u = left ? t / d : -t * l / q;
            mild = left || or_mild(l);
        } else if (l > 0.0) {
            f = left ? d : pow(l, d);
            g = left ? pow(l, d - 1.0) : log(l);
            u = t * f * g;
            mild = or_mild(f);
        }
        if (!isfinite(f) || !isfinite(g)) {
            o.ev |= OR_WILD << r;
            u = 1.0;
        } else if (f == 0.0 || (g == 0.0 && mild)) {
            o.ev |= OR_ZERO << r;
            u = 1.0;
        } else if (!mild || !or_in_range(u)) {
            o.ev |= OR_REDO;
        }
        o.t[r] = u;
    }
    return o;
}

__device__ __forceinline__ OrDual or_dual(const uint32_t *__restrict__ rec, int m,
                                          const double *__restrict__ c, int j, const OrRows &R,
                                          const int (&q)[2])
{
    dv16 S0, S1;
    OrDual t = {{0.0, 0.0}, {0.0, 0.0}, 0};
    int ev = 0;                       /* of the path so far */
    int least[2] = {0, 0}, most[2] = {0, 0}; /* exponents since the last start */
    int sp = -1; /* entries below the top; -1: empty */
    for (int i = 0; i < m; ++i) {
        const uint4 w = ((const uint4 *)rec)[i]; /* operator, children, slot */
        const uint32_t op = w.x;
        if (op == OP_CONST || op == OP_VAR) {
            if (sp >= 0) {
                S0[sp] = t.v[0];
                S0[sp + 8] = t.t[0];
                S1[sp] = t.v[1];
                S1[sp + 8] = t.t[1];
            }
            ++sp;
            if (op == OP_CONST) {
                t.v[0] = t.v[1] = c[w.w];
                t.t[0] = t.t[1] = (int)w.w == j ? 1.0 : 0.0;
            } else {
                const double *col = R.cols64 + (size_t)w.w * (size_t)R.n;
                t.v[0] = col[q[0]];
                t.v[1] = col[q[1]];
                t.t[0] = t.t[1] = 0.0;
            }
            continue;
        }
        if (op == OP_ADD || op == OP_SUB) { /* the tangent as it is */
            --sp;
            const double av[2] = {S0[sp], S1[sp]}, at[2] = {S0[sp + 8], S1[sp + 8]};
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                t.v[r] = op == OP_ADD ? av[r] + t.v[r] : av[r] - t.v[r];
                t.t[r] = op == OP_ADD ? at[r] + t.t[r] : at[r] - t.t[r];
            }
            continue;
        }
        if (ft_is_binary(op)) {
            --sp;
            const double av[2] = {S0[sp], S1[sp]}, at[2] = {S0[sp + 8], S1[sp + 8]};
            const int left = at[0] != 0.0 || at[1] != 0.0; /* the path's side */
            if (op == OP_MUL) {
                t.ev = 0;
                if (left || t.t[0] != 0.0 || t.t[1] != 0.0) {
#pragma unroll
                    for (int r = 0; r < 2; ++r)
                        t.t[r] = or_tan(left ? t.v[r] : av[r], left ? at[r] : t.t[r], r, t.ev);
                }
#pragma unroll
                for (int r = 0; r < 2; ++r) t.v[r] = av[r] * t.v[r];
            } else {
                t = or_divide_or_pow(op, av[0], av[1], t.v[0], t.v[1], left ? at[0] : t.t[0],
                                     left ? at[1] : t.t[1], left);
            }
        } else {
            t = or_unary(op, t.v[0], t.v[1], t.t[0], t.t[1]);
        }
        ev |= t.ev & OR_REDO;
        if (t.t[0] == 0.0 && t.t[1] == 0.0) continue; /* off the path */
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const int what = t.ev & ((OR_ZERO | OR_WILD) << r);
            const int e = __builtin_amdgcn_frexp_exp(t.t[r]); /* 0 off the path */
            if (what) {
                ev = (ev & ~((OR_ZERO | OR_WILD) << r)) | what;
                least[r] = most[r] = 0;
            } else {
                least[r] = min(least[r], e);
                most[r] = max(most[r], e);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const int e = __builtin_amdgcn_frexp_exp(t.t[r]);
        if (e - least[r] > OR_ADJOINT || most[r] - e > OR_ADJOINT) ev |= OR_REDO;
        if (ev & (OR_ZERO << r)) t.t[r] = 0.0;
        if (ev & (OR_WILD << r)) ev |= OR_REDO;
    }
    t.ev = ev & OR_REDO;
    return t;
}

/* One tile of a maximum scan: max |r| with its lowest row and, with LEVEL, the
   interval of steps along the segment's constant (mx_scan_kernel's rules). */
template <bool LEVEL>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(LEVEL ? 2 : 3))) void or_max_kernel(
    const int *__restrict__ segs, const OrSet *__restrict__ sets, const uint32_t *__restrict__ code,
    const uint32_t *__restrict__ prog, const double *__restrict__ c0, int kmax, int ntrials,
    const int *__restrict__ coords, const double *__restrict__ levels, OrRows R,
    OrMax *__restrict__ part, int tiles, int tile_rows, int *__restrict__ redo)
{
    constexpr int RR = LEVEL ? 2 : 4;
    const int li = blockIdx.x / tiles, tile = blockIdx.x - li * tiles;
    const int seg = segs[li];
    const OrSet d = sets[seg / ntrials];
    const double *cst = c0 + (size_t)seg * (size_t)kmax;
    const int lane = threadIdx.x;
    const int begin = tile * tile_rows, end = min(R.n, begin + tile_rows);
    const int coord = LEVEL ? coords[seg] : -1;
    const double level = LEVEL ? levels[seg] : 0.0;
    unsigned long long key = 0ull;
    int at = 0x7fffffff, bad = 0, veto = 0;
    double lo = -__builtin_inf(), hi = __builtin_inf();
    for (int base = begin; base < end; base += 64 * RR) {
        int q[RR];
#pragma unroll
        for (int r = 0; r < RR; ++r) q[r] = min(base + 64 * r + lane, R.n - 1);
        double pred[RR], b[RR];
        if constexpr (LEVEL) {
            const OrDual o = or_dual(prog + d.r_off, d.m, cst, coord, R, q);
#pragma unroll
            for (int r = 0; r < RR; ++r) {
                pred[r] = o.v[r];
                b[r] = o.t[r];
            }
            bad |= o.ev;
        } else {
            const vm_d4 o = or_value((const uint2 *)(code + d.t_off), d.t_m, cst, R, q);
#pragma unroll
            for (int r = 0; r < RR; ++r) {
                pred[r] = o[r];
                b[r] = 0.0;
            }
        }
#pragma unroll
        for (int r = 0; r < RR; ++r) {
            const int row = base + 64 * r + lane;
            if (row >= end) continue;
            const double rr = pred[r] - R.y64[row];
            if (or_bad_row(pred[r], rr)) {
                bad = 1;
                continue;
            }
            /* A lane's rows come in increasing order: the first of equal
               maxima stays. */
            const unsigned long long k = (unsigned long long)__double_as_longlong(fabs(rr));
            if (k > key || at == 0x7fffffff) {
                key = k;
                at = row;
            }
            if (!LEVEL) continue;
            if (b[r] == 0.0) {
                veto |= fabs(rr) > level;
            } else {
                const double e1 = (-level - rr) / b[r];
                const double e2 = (level - rr) / b[r];
                lo = fmax(lo, fmin(e1, e2));
                hi = fmin(hi, fmax(e1, e2));
            }
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long k = __shfl_xor(key, o, 64);
        const int a = __shfl_xor(at, o, 64);
        if (k > key || (k == key && a < at)) {
            key = k;
            at = a;
        }
        if (LEVEL) {
            lo = fmax(lo, __shfl_xor(lo, o, 64));
            hi = fmin(hi, __shfl_xor(hi, o, 64));
        }
    }
    const int anyveto = __any(veto) ? 1 : 0;
    const int anybad = __any(bad) ? 1 : 0;
    if (lane == 0) {
        part[(size_t)li * (size_t)tiles + (size_t)tile] = {key, lo, hi, at, anyveto};
        if (anybad) redo[seg] = 1;
    }
}

} /* namespace */

/* Rows of a tile: a value does not depend on it.  Eight steps of 256 rows
   where that still makes four waves for each of the 1024 SIMDs, else two. */
int or_max_tiles(int n, int nsegs, int *tile_rows)
{
    *tile_rows = (long long)nsegs * ((n + 2047) / 2048) >= 4096 ? 2048 : 512;
    return (n + *tile_rows - 1) / *tile_rows;
}

void or_launch_keys(bool rank, int nlist, hipStream_t s, const int *segs, const OrSet *sets,
                    const uint32_t *code, const double *c0, int kmax, int ntrials, OrRows rows,
                    unsigned long long *keys, uint32_t *row_of, int *status)
{
    if (nlist <= 0) return;
    int tile_rows;
    const int tiles = or_max_tiles(rows.n, nlist, &tile_rows);
    const unsigned grid = (unsigned)nlist * (unsigned)tiles;
    if (rank)
        or_keys_kernel<true><<<grid, 64, 0, s>>>(segs, sets, code, c0, kmax, ntrials, rows, tiles,
                                                 tile_rows, keys, row_of, status);
    else
        or_keys_kernel<false><<<grid, 64, 0, s>>>(segs, sets, code, c0, kmax, ntrials, rows, tiles,
                                                  tile_rows, keys, row_of, status);
}

void or_launch_max(bool level, int nlist, hipStream_t s, const int *segs, const OrSet *sets,
                   const uint32_t *code, const uint32_t *prog, const double *c0, int kmax,
                   int ntrials, const int *coords, const double *levels, OrRows rows, OrMax *part,
                   int tiles, int tile_rows, int *redo)
{
    if (nlist <= 0) return;
    const unsigned grid = (unsigned)nlist * (unsigned)tiles;
    if (level)
        or_max_kernel<true><<<grid, 64, 0, s>>>(segs, sets, code, prog, c0, kmax, ntrials, coords,
                                                levels, rows, part, tiles, tile_rows, redo);
    else
        or_max_kernel<false><<<grid, 64, 0, s>>>(segs, sets, code, prog, c0, kmax, ntrials, coords,
                                                 levels, rows, part, tiles, tile_rows, redo);
}
