/*
 * Exact order, rank and maximum statistics of candidate predictions on
 * gfx950: the device stages behind rc_order_stat_score_batch,
 * rc_rank_score_batch and rc_max_scan_batch (reference eval.cu:2888-3133,
 * 4093-4850).
 *
 * Every call scores nsets x ntrials segments: segment seg = set * ntrials +
 * trial evaluates set `set`'s post-order fit records (the rc_fit_batch
 * program form) over the resident f64 rows with the constants c0[seg * kmax
 * ...], in f64.  The statistics are exact functions of the multiset of
 * values (median, maximum) or of integer ranks (rank sums), so they do not
 * depend on how the work is split; the interquartile mean is summed left to
 * right over the sorted window, the CPU's order, so it agrees bit for bit.
 *
 * MI355X layout:
 *  - the row kernels of rc_order_kern.hip evaluate the records and write one
 *    64-bit sort key (and the row, for ranks), or a tile's maximum; programs
 *    that do not fit their registers run here, one thread per (segment, row)
 *    with a private value array;
 *  - the median is a selection: one workgroup per segment narrows the range of
 *    keys that holds the middle ones by histograms of its leading bits;
 *  - rocPRIM's segmented radix sort (through hipCUB) orders each segment for
 *    the interquartile mean, summed by one wave per segment, and for ranks;
 *  - average ranks come from two scans per segment in one workgroup: a
 *    forward max-scan finds each position's tie-run start, a backward
 *    min-scan its run end, and A = start + end - n is the doubled centred
 *    rank; its products with the target's cached ranks accumulate in exact
 *    128-bit integers (two 64-bit halves), so the reduction order is free;
 *  - the maximum scan reduces an integer key (|r| bit patterns order like the
 *    values), the lowest maximising row and the feasibility interval of a level
 *    along one constant, over tiles and then over a segment's tiles.
 */
#include "rc_fit_dev.h"
#include "rc_block.h"
#include "rc_fitvm.h"
#include "rc_internal.h"
#include "rc_order_kern.h"

#include <hipcub/hipcub.hpp>

#include <string.h>

#include <math.h>

#include <algorithm>
#include <vector>

extern "C" int rch_fitvm_compile(const unsigned int *rec, int words, int p, int nvars, int col_bytes,
                                 unsigned int flags, unsigned int *fwd, int cap_f,
                                 unsigned int *rev, int cap_r, int *info);

namespace {

constexpr int RK_THREADS = 256;
constexpr int MX_THREADS = 256;
constexpr unsigned long long KEY_BAD = 0xFFFFFFFFFFFFFFFFull;

/* Order-preserving 64-bit key of a finite f64 (-0.0 keyed as +0.0, so the two
   form one tie, as f64 == has them). */
__device__ __forceinline__ unsigned long long rk_key(double v)
{
    if (v == 0.0) v = 0.0;
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}

__device__ __forceinline__ double os_value(unsigned long long k)
{
    return __longlong_as_double((long long)k);
}

/* Prediction of (segment, row): the records of the segment's set with the
   segment's constants. */
__device__ __forceinline__ double seg_predict(const uint32_t *__restrict__ prog,
                                              const uint32_t *__restrict__ off,
                                              const double *__restrict__ c0, int kmax,
                                              const double *__restrict__ cols64, int n, int seg,
                                              int ntrials, int row, double *v)
{
    const int set = seg / ntrials;
    const uint32_t *nd = prog + off[set];
    const int m = (int)((off[set + 1] - off[set]) / 4u);
    ft_rec_values(nd, m, cols64, n, row, c0 + (size_t)seg * (size_t)kmax, v);
    return v[m - 1];
}

/* Sort keys of every (listed segment, row): |pred - y| bit patterns (order
   statistics, eval.cu:4383-4419) or rank keys of pred with the row as the
   payload (ranks, eval.cu:2952-2982).  A non-finite value keys last and
   flags its segment (status 2). */
template <bool RANK>
__global__ __launch_bounds__(256) void os_keys_kernel(
    const uint32_t *__restrict__ prog, const uint32_t *__restrict__ off,
    const double *__restrict__ c0, int kmax, const double *__restrict__ cols64,
    const double *__restrict__ y64, int n, const int *__restrict__ segs, int nlist, int ntrials,
    unsigned long long *__restrict__ keys, uint32_t *__restrict__ rows, int *__restrict__ status)
{
    const long long total = (long long)n * (long long)nlist;
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long u = (long long)blockIdx.x * blockDim.x + threadIdx.x; u < total; u += stride) {
        const int li = (int)(u / n);
        const int row = (int)(u - (long long)li * n);
        const int seg = segs[li];
        const long long i = (long long)seg * n + row;
        double v[FT_MAX_NODES];
        const double pred = seg_predict(prog, off, c0, kmax, cols64, n, seg, ntrials, row, v);
        if (RANK) {
            if (!isfinite(pred)) {
                keys[i] = KEY_BAD;
                status[seg] = 2;
            } else {
                keys[i] = rk_key(pred);
            }
            rows[i] = (uint32_t)row;
        } else {
            const double r = pred - y64[row];
            if (!isfinite(pred) || fabs(pred) > 1e30 || !isfinite(r)) {
                keys[i] = KEY_BAD;
                status[seg] = 2;
            } else {
                keys[i] = (unsigned long long)__double_as_longlong(fabs(r));
            }
        }
    }
}

/* Rank keys of the target (one segment). */
__global__ void rk_target_keys_kernel(const double *__restrict__ y64, int n,
                                      unsigned long long *__restrict__ keys,
                                      uint32_t *__restrict__ rows, int *__restrict__ bad)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double v = y64[i];
    if (!isfinite(v)) {
        keys[i] = KEY_BAD;
        *bad = 1;
    } else {
        keys[i] = rk_key(v);
    }
    rows[i] = (uint32_t)i;
}

/* The median of one segment's unsorted keys (metrics.rs:1193-1208), by
   selection.  The keys that can be the lower middle one lie in [base, base +
   range]; a histogram of their leading 11 bits says in which bin, which is the
   next range, until a bin has no more than SEL_CAP keys: those are gathered and
   sorted in LDS.  The upper middle key is the next of them, or the least key
   above the last range.  Two to three passes over the keys in all, each at the
   rate one CU reads, where the full sort made eight and wrote as much: 256
   segments of 262 144 keys take 0.30 ms, their sort 9.1. */
constexpr int SEL_THREADS = 1024;
constexpr int SEL_BINS = 2048;
constexpr int SEL_CAP = 4096;
__global__ __launch_bounds__(SEL_THREADS) void os_select_kernel(
    const unsigned long long *__restrict__ keys, int n, int nsegs, double *__restrict__ out,
    const int *__restrict__ status)
{
    __shared__ unsigned int hist[SEL_BINS];
    __shared__ unsigned int wsum[SEL_THREADS / 64];
    __shared__ unsigned long long buf[SEL_CAP];
    __shared__ unsigned long long wa[SEL_THREADS / 64], wb[SEL_THREADS / 64];
    __shared__ unsigned int sh_n;
    __shared__ int sh_bin;
    __shared__ unsigned int sh_before;
    const int seg = blockIdx.x;
    if (seg >= nsegs) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (status[seg] != 0) { /* block-uniform */
        if (tid == 0) out[seg] = __builtin_nan("");
        return;
    }
    const unsigned long long *k = keys + (size_t)seg * (size_t)n;
    /* Every key of the segment, four loads in flight a thread. */
    auto each = [&](auto &&f) {
        const unsigned int m = (unsigned int)n;
        for (unsigned int i0 = tid; i0 < m; i0 += 4u * SEL_THREADS) {
            unsigned long long v[4];
#pragma unroll
            for (unsigned int u = 0; u < 4u; ++u) v[u] = k[min(i0 + u * SEL_THREADS, m - 1u)];
#pragma unroll
            for (unsigned int u = 0; u < 4u; ++u)
                if (i0 + u * SEL_THREADS < m) f(v[u]);
        }
    };
    /* The block's least a and greatest b, in every thread. */
    auto ends = [&](unsigned long long &a, unsigned long long &b) {
        for (int o = 32; o > 0; o >>= 1) {
            const unsigned long long x = __shfl_xor(a, o, 64), y = __shfl_xor(b, o, 64);
            a = x < a ? x : a;
            b = y > b ? y : b;
        }
        if (lane == 0) {
            wa[wave] = a;
            wb[wave] = b;
        }
        __syncthreads();
        for (int w = 0; w < SEL_THREADS / 64; ++w) {
            a = wa[w] < a ? wa[w] : a;
            b = wb[w] > b ? wb[w] : b;
        }
        __syncthreads();
    };
    unsigned long long least = KEY_BAD, most = 0ull;
    each([&](unsigned long long v) {
        least = v < least ? v : least;
        most = v > most ? v : most;
    });
    ends(least, most);
    unsigned long long base = least, range = most - least;
    unsigned int rank = (unsigned int)((n - 1) / 2), count = (unsigned int)n;
    while (range != 0ull && count > SEL_CAP) {
        const int bits = 64 - __clzll((long long)range);
        const int shift = bits > 11 ? bits - 11 : 0;
        for (int i = tid; i < SEL_BINS; i += SEL_THREADS) hist[i] = 0u;
        __syncthreads();
        each([&](unsigned long long v) {
            const unsigned long long d = v - base; /* below base: wraps past range */
            if (d <= range) atomicAdd(&hist[(unsigned int)(d >> shift)], 1u);
        });
        __syncthreads();
        /* The bin that holds `rank`: a scan of two bins a thread. */
        const unsigned int h0 = hist[2 * tid], h1 = hist[2 * tid + 1];
        unsigned int run = h0 + h1;
        for (int o = 1; o < 64; o <<= 1) {
            const unsigned int x = __shfl_up(run, o, 64);
            if (lane >= o) run += x;
        }
        if (lane == 63) wsum[wave] = run;
        __syncthreads();
        for (int w = 0; w < wave; ++w) run += wsum[w];
        const unsigned int before = run - h0 - h1;
        if (rank >= before && rank < before + h0) {
            sh_bin = 2 * tid;
            sh_before = before;
        } else if (rank >= before + h0 && rank < run) {
            sh_bin = 2 * tid + 1;
            sh_before = before + h0;
        }
        __syncthreads();
        const unsigned long long start = (unsigned long long)sh_bin << shift;
        count = hist[sh_bin];
        rank -= sh_before;
        base += start;
        const unsigned long long width = (1ull << shift) - 1ull, rest = range - start;
        range = width < rest ? width : rest;
        __syncthreads();
    }
    /* The keys of the last range into LDS (one value of them where it is a
       single key), and the least key above it. */
    if (tid == 0) sh_n = 0u;
    __syncthreads();
    unsigned long long above = KEY_BAD, unused = 0ull;
    const unsigned long long last = base + range;
    each([&](unsigned long long v) {
        if (v > last) above = v < above ? v : above;
        else if (range != 0ull && v >= base) buf[atomicAdd(&sh_n, 1u)] = v;
    });
    ends(above, unused);
    unsigned long long low = base, high = base;
    if (range != 0ull) {
        const unsigned int m = sh_n; /* = count <= SEL_CAP */
        unsigned int p2 = 2u;
        while (p2 < m) p2 <<= 1;
        for (unsigned int i = m + tid; i < p2; i += SEL_THREADS) buf[i] = KEY_BAD;
        __syncthreads();
        for (unsigned int size = 2u; size <= p2; size <<= 1)
            for (unsigned int step = size >> 1; step > 0u; step >>= 1) {
                for (unsigned int t = tid; t < p2 / 2u; t += SEL_THREADS) {
                    const unsigned int i = 2u * t - (t & (step - 1u)), j = i + step;
                    const bool up = (i & size) == 0u;
                    const unsigned long long x = buf[i], y = buf[j];
                    if ((x > y) == up) {
                        buf[i] = y;
                        buf[j] = x;
                    }
                }
                __syncthreads();
            }
        low = buf[rank];
        high = rank + 1u < m ? buf[rank + 1u] : above;
    } else if (rank + 1u >= count) {
        high = above;
    }
    if (tid == 0) out[seg] = (n & 1) ? os_value(low) : 0.5 * (os_value(low) + os_value(high));
}

/* The interquartile mean of one sorted segment (metrics.rs:1209-1223): one
   wave per segment; the window is summed left to right, the CPU's order, from
   blocks that the wave has staged in LDS while the previous one is summed (a
   chain of dependent f64 adds; one lane that loaded each value itself waited
   on memory for every one: 256 segments of 262 144 keys 8.5 ms, now 0.74). */
constexpr int MEAN_BLOCK = 1024;
__global__ __launch_bounds__(64) void os_mean_kernel(const unsigned long long *__restrict__ keys,
                                                     int n, int nsegs, double *__restrict__ out,
                                                     const int *__restrict__ status)
{
    __shared__ __align__(16) double stage[MEAN_BLOCK];
    const int seg = blockIdx.x;
    if (seg >= nsegs) return;
    const int lane = threadIdx.x;
    if (status[seg] != 0) { /* wave-uniform */
        if (lane == 0) out[seg] = __builtin_nan("");
        return;
    }
    const unsigned long long *k = keys + (size_t)seg * (size_t)n;
    int lo = 0, hi = n;
    if (n >= 4) {
        lo = n / 4;
        hi = max((3 * n) / 4, lo + 1);
    }
    constexpr int PER = MEAN_BLOCK / 64;
    unsigned long long v[PER];
    auto load = [&](int at) {
#pragma unroll
        for (int u = 0; u < PER; ++u) v[u] = k[min(at + 64 * u + lane, n - 1)];
    };
    double s = 0.0;
    load(lo);
    for (int at = lo; at < hi; at += MEAN_BLOCK) {
        __syncthreads();
#pragma unroll
        for (int u = 0; u < PER; ++u) stage[64 * u + lane] = os_value(v[u]);
        __syncthreads();
        if (at + MEAN_BLOCK < hi) load(at + MEAN_BLOCK);
        const int m = min(MEAN_BLOCK, hi - at);
        int i = 0;
        for (; i + 16 <= m; i += 16) {
            double w[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) w[u] = stage[i + u];
#pragma unroll
            for (int u = 0; u < 16; ++u) s += w[u];
        }
        for (; i < m; ++i) s += stage[i];
    }
    if (lane == 0) out[seg] = s / (double)(hi - lo);
}

/* ---- exact 128-bit accumulation ------------------------------------------- */

struct I128 {
    unsigned long long hi, lo;
};

__device__ __forceinline__ void i128_add(I128 &a, const I128 &b)
{
    const unsigned long long lo = a.lo + b.lo;
    a.hi += b.hi + (lo < a.lo ? 1ull : 0ull);
    a.lo = lo;
}

/* Add a signed 64-bit value, sign-extended. */
__device__ __forceinline__ void i128_add64(I128 &a, long long v)
{
    I128 b = {v < 0 ? ~0ull : 0ull, (unsigned long long)v};
    i128_add(a, b);
}

/* Workgroup sum of one I128 per thread (exact, so any order). */
template <int T>
__device__ __forceinline__ I128 i128_block_sum(I128 v, I128 *sh)
{
    const int tid = threadIdx.x;
    sh[tid] = v;
    __syncthreads();
    for (int s = T / 2; s > 0; s >>= 1) {
        if (tid < s) {
            I128 a = sh[tid];
            i128_add(a, sh[tid + s]);
            sh[tid] = a;
        }
        __syncthreads();
    }
    const I128 r = sh[0];
    __syncthreads();
    return r;
}

/* ---- average ranks by two scans -------------------------------------------- */

struct MaxCarry {
    int run;
    __device__ int operator()(int block_aggregate)
    {
        const int old = run;
        run = max(run, block_aggregate);
        return old;
    }
};

struct MinCarry {
    int run;
    __device__ int operator()(int block_aggregate)
    {
        const int old = run;
        run = min(run, block_aggregate);
        return old;
    }
};

/* For each sorted segment: pass 1 stores every position's tie-run start
   (the last position <= i whose key differs from its predecessor); pass 2
   walks the segment backwards for the run end and forms the doubled centred
   rank A = start + end + 1 - n (metrics.rs:1258-1286: run [s, e) gets
   s + e - n).  TARGET: write B[row] = A and Sigma B^2; otherwise accumulate
   Sigma A * B[row] and Sigma A^2 into out[4 seg ..] (hi, lo, hi, lo). */
template <bool TARGET>
__global__ __launch_bounds__(RK_THREADS) void rk_runs_kernel(
    const unsigned long long *__restrict__ keys, const uint32_t *__restrict__ rows, int n,
    int nsegs, int *__restrict__ start_of, long long *__restrict__ B,
    unsigned long long *__restrict__ out)
{
    typedef hipcub::BlockScan<int, RK_THREADS> Scan;
    __shared__ typename Scan::TempStorage tmp;
    __shared__ I128 red[RK_THREADS];
    const int seg = blockIdx.x;
    if (seg >= nsegs) return;
    const int tid = threadIdx.x;
    const size_t base = (size_t)seg * (size_t)n;
    const unsigned long long *k = keys + base;
    const uint32_t *rw = rows + base;
    int *st = start_of + base;

    MaxCarry mc = {0};
    for (int c0 = 0; c0 < n; c0 += RK_THREADS) {
        const int i = c0 + tid;
        int f = 0;
        if (i < n) f = (i == 0 || k[i] != k[i - 1]) ? i : 0;
        int s;
        Scan(tmp).InclusiveScan(f, s, hipcub::Max(), mc);
        __syncthreads();
        if (i < n) st[i] = s;
    }
    __syncthreads();

    I128 ab = {0ull, 0ull}, aa = {0ull, 0ull};
    MinCarry nc = {0x7fffffff};
    for (int c0 = ((n - 1) / RK_THREADS) * RK_THREADS; c0 >= 0; c0 -= RK_THREADS) {
        /* Thread t takes position c0 + (T - 1 - t): an inclusive scan over
           threads is then a suffix scan over positions. */
        const int i = c0 + (RK_THREADS - 1 - tid);
        int f = 0x7fffffff;
        if (i < n) f = (i == n - 1 || k[i] != k[i + 1]) ? i : 0x7fffffff;
        int e;
        Scan(tmp).InclusiveScan(f, e, hipcub::Min(), nc);
        __syncthreads();
        if (i < n) {
            const long long A = (long long)st[i] + (long long)e + 1 - (long long)n;
            if (TARGET) {
                B[rw[i]] = A;
                i128_add64(aa, A * A);
            } else {
                i128_add64(ab, A * B[rw[i]]);
                i128_add64(aa, A * A);
            }
        }
    }
    if (!TARGET) ab = i128_block_sum<RK_THREADS>(ab, red);
    aa = i128_block_sum<RK_THREADS>(aa, red);
    if (tid == 0) {
        if (TARGET) {
            out[0] = aa.hi;
            out[1] = aa.lo;
        } else {
            out[4 * (size_t)seg + 0] = ab.hi;
            out[4 * (size_t)seg + 1] = ab.lo;
            out[4 * (size_t)seg + 2] = aa.hi;
            out[4 * (size_t)seg + 3] = aa.lo;
        }
    }
}

/* ---- the exact maximum-error scan ----------------------------------------- */

/* One workgroup per segment marked in redo, those that the row kernels do not
   run and those in which they met a row or a derivative that is not finite or
   may have left the range of f64 on its way (eval.cu:4505-4600): max |r| as an integer
   max of bit patterns with the lowest row on ties; with a constant `coord`
   and a finite level t >= 0, the intersection of the per-row intervals
   {delta : |r_i + b_i delta| <= t}, b_i = d pred_i / d c_coord from the f64
   adjoint sweep (rows with b_i == 0 only veto). */
__global__ __launch_bounds__(MX_THREADS) void mx_scan_kernel(
    const uint32_t *__restrict__ prog, const uint32_t *__restrict__ off,
    const int *__restrict__ pcount, const double *__restrict__ c0, int kmax,
    const int *__restrict__ coords, const double *__restrict__ levels,
    const double *__restrict__ cols64, const double *__restrict__ y64, int n, int nsegs,
    int ntrials, const int *__restrict__ redo, RcMaxOut *__restrict__ out)
{
    __shared__ unsigned long long skey[MX_THREADS];
    __shared__ int srow[MX_THREADS];
    __shared__ double slo[MX_THREADS];
    __shared__ double shi[MX_THREADS];
    __shared__ int sbad[MX_THREADS];
    const int seg = blockIdx.x;
    if (seg >= nsegs || !redo[seg]) return;
    const int tid = threadIdx.x;
    const int set = seg / ntrials;
    const uint32_t *nd = prog + off[set];
    const int m = (int)((off[set + 1] - off[set]) / 4u);
    const int p = pcount[set];
    const double *c = c0 + (size_t)seg * (size_t)kmax;
    const int coord = (p > 0 && coords[seg] >= 0 && coords[seg] < p) ? coords[seg] : -1;
    const double level = levels[seg];
    const bool want = coord >= 0 && isfinite(level) && level >= 0.0;

    unsigned long long mykey = 0ull;
    int myrow = 0x7fffffff;
    double mylo = -__builtin_inf(), myhi = __builtin_inf();
    int mybad = 0; /* bit 0: a non-finite row; bit 1: the level is vetoed */
    for (int row = tid; row < n; row += MX_THREADS) {
        double v[FT_MAX_NODES];
        ft_rec_values(nd, m, cols64, n, row, c, v);
        const double pred = v[m - 1];
        const double r = pred - y64[row];
        if (!isfinite(pred) || fabs(pred) > 1e30 || !isfinite(r)) {
            mybad |= 1;
            break;
        }
        const unsigned long long key = (unsigned long long)__double_as_longlong(fabs(r));
        if (key > mykey || (key == mykey && row < myrow)) {
            mykey = key;
            myrow = row;
        }
        if (want && !(mybad & 2)) {
            double adj[FT_MAX_NODES];
            double g[FT_KMAX];
            ft_rec_gradient(nd, m, v, adj, g, p);
            const double b = g[coord];
            if (!isfinite(b)) {
                mybad |= 1;
                break;
            }
            if (b == 0.0) {
                if (fabs(r) > level) mybad |= 2;
            } else {
                const double e1 = (-level - r) / b;
                const double e2 = (level - r) / b;
                mylo = fmax(mylo, fmin(e1, e2));
                myhi = fmin(myhi, fmax(e1, e2));
            }
        }
    }
    skey[tid] = mykey;
    srow[tid] = myrow;
    slo[tid] = mylo;
    shi[tid] = myhi;
    sbad[tid] = mybad;
    __syncthreads();
    for (int s = MX_THREADS / 2; s > 0; s >>= 1) {
        if (tid < s) {
            const int j = tid + s;
            if (skey[j] > skey[tid] || (skey[j] == skey[tid] && srow[j] < srow[tid])) {
                skey[tid] = skey[j];
                srow[tid] = srow[j];
            }
            slo[tid] = fmax(slo[tid], slo[j]);
            shi[tid] = fmin(shi[tid], shi[j]);
            sbad[tid] |= sbad[j];
        }
        __syncthreads();
    }
    if (tid == 0) {
        const int bad = sbad[0];
        RcMaxOut o;
        o.status = (bad & 1) ? 2 : 0;
        o.vmax = (bad & 1) ? __builtin_nan("") : os_value(skey[0]);
        o.row = (bad & 1) ? -1 : srow[0];
        o.lo = (bad & 2) ? __builtin_inf() : slo[0];
        o.hi = (bad & 2) ? -__builtin_inf() : shi[0];
        out[seg] = o;
    }
}

/* A listed segment's tiles in one: the greatest |r| with its lowest row, the
   intersection of the intervals. */
__global__ __launch_bounds__(64) void mx_finish_kernel(const int *__restrict__ segs, int nlist,
                                                       const OrMax *__restrict__ part, int tiles,
                                                       RcMaxOut *__restrict__ out)
{
    const int li = blockIdx.x;
    if (li >= nlist) return;
    unsigned long long key = 0ull;
    int row = 0x7fffffff, veto = 0;
    double lo = -__builtin_inf(), hi = __builtin_inf();
    for (int t = threadIdx.x; t < tiles; t += 64) {
        const OrMax m = part[(size_t)li * (size_t)tiles + (size_t)t];
        if (m.key > key || (m.key == key && m.row < row)) {
            key = m.key;
            row = m.row;
        }
        lo = fmax(lo, m.lo);
        hi = fmin(hi, m.hi);
        veto |= m.veto;
    }
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long k = __shfl_xor(key, o, 64);
        const int r = __shfl_xor(row, o, 64);
        if (k > key || (k == key && r < row)) {
            key = k;
            row = r;
        }
        lo = fmax(lo, __shfl_xor(lo, o, 64));
        hi = fmin(hi, __shfl_xor(hi, o, 64));
    }
    if (__any(veto)) {
        lo = __builtin_inf();
        hi = -__builtin_inf();
    }
    if (threadIdx.x == 0) {
        RcMaxOut o;
        o.status = 0;
        o.vmax = os_value(key);
        o.row = row;
        o.lo = lo;
        o.hi = hi;
        out[segs[li]] = o;
    }
}

/* ---- host side ------------------------------------------------------------- */

/* A call's inputs on the device, gathered in one host block and sent in one
   copy: programs, constants, value streams, segment lists and what the kernels
   find cleared. */
struct StageInput {
    std::vector<OrSet> sets;
    std::vector<uint32_t> code;
    std::vector<int> fast, general; /* segments by the route of their set */
    uint32_t *prog = nullptr, *off = nullptr, *d_code = nullptr;
    int *pcount = nullptr, *coords = nullptr, *lists = nullptr, *flags = nullptr;
    double *c0 = nullptr, *levels = nullptr;
    OrSet *d_sets = nullptr;
};

/* What the record sweep takes: a canonical post-order tree (each record's
   children are the tops of the evaluation stack) no deeper than its stack. */
bool stack_tree(const unsigned int *nd, int m)
{
    std::vector<uint32_t> st;
    size_t depth = 0;
    for (int i = 0; i < m; ++i) {
        const uint32_t op = nd[4 * i], k0 = nd[4 * i + 1], k1 = nd[4 * i + 2];
        if (op != OP_CONST && op != OP_VAR) {
            const bool two = op == OP_ADD || op == OP_SUB || op == OP_MUL || op == OP_DIV || op == OP_POW;
            if (two) {
                if (st.size() < 2 || st.back() != k1) return false;
                st.pop_back();
            }
            if (st.empty() || st.back() != k0) return false;
            st.pop_back();
        }
        st.push_back((uint32_t)i);
        depth = std::max(depth, st.size());
    }
    return st.size() == 1 && depth <= OR_SDEPTH + 1;
}

/* The sets' records and value streams (none where the program does not fit
   the stream's files). */
void stage_sets(const RcCtx *c, const unsigned int *prog, const unsigned int *off,
                const int *pcount, int nsets, StageInput *in)
{
    uint32_t buf[OR_STREAM_WORDS];
    in->sets.resize((size_t)nsets);
    for (int s = 0; s < nsets; ++s) {
        OrSet &d = in->sets[(size_t)s];
        const int words = (int)(off[s + 1] - off[s]);
        int info[6];
        d.r_off = off[s];
        d.m = words / 4;
        d.t_off = (uint32_t)in->code.size();
        d.t_m = 0;
        if (c->sets[0].n <= OR_MAX_ROWS &&
            rch_fitvm_compile(prog + off[s], words, pcount[s], c->sets[0].v, 8,
                              VMC_INPUTS_IN_U | VMC_VALUE_ONLY | VMC_SMALL_U, buf,
                              OR_STREAM_WORDS, nullptr, 0, info) == 0) {
            d.t_m = info[0];
            in->code.insert(in->code.end(), buf, buf + 2 * info[0]);
        }
    }
}

/* coords / levels: nsegs each, or null; flags: nsegs ints at the device. */
int stage_inputs(RcCtx *c, const unsigned int *prog, const unsigned int *off, const int *pcount,
                 int nsets, int nsegs, int kmax, const double *c0, const int *coords,
                 const double *levels, const std::vector<int> &flags, StageInput *in)
{
    RcOrderBufs &b = c->order;
    std::vector<int> lists(in->fast);
    lists.insert(lists.end(), in->general.begin(), in->general.end());
    const size_t ns = (size_t)nsegs;
    const size_t words = off[nsets];
    RcBlock h(b.h_in, 4 * words + 8 * ns * (size_t)(kmax + 3) + 64 * (size_t)nsets +
                          4 * in->code.size() + 4096);
    const size_t o_prog = h.put(prog, 4 * words);
    const size_t o_off = h.put(off, 4 * ((size_t)nsets + 1));
    const size_t o_pc = h.put(pcount, 4 * (size_t)nsets);
    const size_t o_c0 = h.put(c0, 8 * ns * (size_t)kmax);
    const size_t o_code = h.put(in->code);
    const size_t o_sets = h.put(in->sets);
    const size_t o_list = h.put(lists);
    const size_t o_flag = h.put(flags);
    const size_t o_co = h.put(coords, coords ? 4 * ns : 0);
    const size_t o_lv = h.put(levels, levels ? 8 * ns : 0);
    const size_t bytes = b.h_in.size();
    if (rc_grow(c, (void **)&b.in, &b.in_cap, bytes, 1) != 0 ||
        hipMemcpyAsync(b.in, b.h_in.data(), bytes, hipMemcpyHostToDevice, c->s_fit) != hipSuccess)
        return -1;
    in->prog = (uint32_t *)(b.in + o_prog);
    in->off = (uint32_t *)(b.in + o_off);
    in->pcount = (int *)(b.in + o_pc);
    in->c0 = (double *)(b.in + o_c0);
    in->d_code = (uint32_t *)(b.in + o_code);
    in->d_sets = (OrSet *)(b.in + o_sets);
    in->lists = (int *)(b.in + o_list);
    in->flags = (int *)(b.in + o_flag);
    in->coords = coords ? (int *)(b.in + o_co) : nullptr;
    in->levels = levels ? (double *)(b.in + o_lv) : nullptr;
    return 0;
}

/* Segment offsets 0, n, 2n, ... for the segmented sort (the host copy stays
   alive with the context, so the asynchronous upload never reads freed
   memory). */
int segment_offsets(RcCtx *c, int nsegs, int n)
{
    std::vector<int> &h = c->order.h_seg;
    h.resize((size_t)nsegs + 1);
    for (int s = 0; s <= nsegs; ++s) h[s] = s * n;
    RcOrderBufs &b = c->order;
    if (rc_grow(c, (void **)&b.seg, &b.seg_cap, h.size(), sizeof(int)) != 0) return -1;
    return hipMemcpyAsync(b.seg, h.data(), sizeof(int) * h.size(), hipMemcpyHostToDevice,
                          c->s_fit) == hipSuccess
               ? 0
               : -1;
}

/* Buffers for `total` keys: to be sorted, or not; with row payloads when
   `pairs`. */
int sort_buffers(RcCtx *c, long long total, bool sorted, bool pairs)
{
    RcOrderBufs &b = c->order;
    const size_t t = (size_t)total;
    if (rc_grow(c, (void **)&b.keys, &b.keys_cap, t, sizeof(unsigned long long)) != 0) return -1;
    if (sorted &&
        rc_grow(c, (void **)&b.keys_out, &b.keys_out_cap, t, sizeof(unsigned long long)) != 0)
        return -1;
    if (pairs &&
        (rc_grow(c, (void **)&b.rows, &b.rows_cap, t, sizeof(uint32_t)) != 0 ||
         rc_grow(c, (void **)&b.rows_out, &b.rows_out_cap, t, sizeof(uint32_t)) != 0 ||
         rc_grow(c, (void **)&b.start_of, &b.start_cap, t, sizeof(int)) != 0))
        return -1;
    return 0;
}

int segmented_sort(RcCtx *c, long long total, int nsegs, bool pairs)
{
    RcOrderBufs &b = c->order;
    size_t need = 0;
    hipError_t e;
    if (pairs)
        e = hipcub::DeviceSegmentedRadixSort::SortPairs(nullptr, need, b.keys, b.keys_out, b.rows,
                                                        b.rows_out, (int)total, nsegs, b.seg,
                                                        b.seg + 1, 0, 64, c->s_fit);
    else
        e = hipcub::DeviceSegmentedRadixSort::SortKeys(nullptr, need, b.keys, b.keys_out, (int)total,
                                                       nsegs, b.seg, b.seg + 1, 0, 64, c->s_fit);
    if (e != hipSuccess) return -1;
    if (rc_grow(c, (void **)&b.temp, &b.temp_cap, need > 0 ? need : 1, 1) != 0) return -1;
    size_t tb = b.temp_cap;
    if (pairs)
        e = hipcub::DeviceSegmentedRadixSort::SortPairs(b.temp, tb, b.keys, b.keys_out, b.rows,
                                                        b.rows_out, (int)total, nsegs, b.seg,
                                                        b.seg + 1, 0, 64, c->s_fit);
    else
        e = hipcub::DeviceSegmentedRadixSort::SortKeys(b.temp, tb, b.keys, b.keys_out, (int)total,
                                                       nsegs, b.seg, b.seg + 1, 0, 64, c->s_fit);
    return e == hipSuccess ? 0 : -1;
}

unsigned grid_for(long long total)
{
    long long blocks = (total + 255) / 256;
    if (blocks > 65535) blocks = 65535;
    return (unsigned)(blocks < 1 ? 1 : blocks);
}

/* The sort keys of every segment: value streams where the set has one, the
   general kernel for the others. */
int launch_keys(RcCtx *c, bool rank, const StageInput &in, int kmax, int ntrials, int *status)
{
    RcRows *r = &c->sets[0];
    RcOrderBufs &b = c->order;
    const int nf = (int)in.fast.size(), ng = (int)in.general.size();
    or_launch_keys(rank, nf, c->s_fit, in.lists, in.d_sets, in.d_code, in.c0, kmax, ntrials,
                   {r->cols64, r->y64, r->n, r->v}, b.keys, b.rows, status);
    if (ng > 0) {
        const unsigned grid = grid_for((long long)r->n * ng);
        if (rank)
            os_keys_kernel<true><<<grid, 256, 0, c->s_fit>>>(
                in.prog, in.off, in.c0, kmax, r->cols64, r->y64, r->n, in.lists + nf, ng, ntrials,
                b.keys, b.rows, status);
        else
            os_keys_kernel<false><<<grid, 256, 0, c->s_fit>>>(
                in.prog, in.off, in.c0, kmax, r->cols64, r->y64, r->n, in.lists + nf, ng, ntrials,
                b.keys, nullptr, status);
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

/* The target's doubled centred ranks B (cached until the f64 rows change)
   and Sigma B^2. */
int rank_prepare(RcCtx *c)
{
    RcOrderBufs &b = c->order;
    if (b.rank_ready) return 0;
    RcRows *r = &c->sets[0];
    const int n = r->n;
    if (n <= 1 || rc_rows_ensure_f64(c, r) != 0) return -1;
    if (sort_buffers(c, n, true, true) != 0 || segment_offsets(c, 1, n) != 0) return -1;
    if (rc_grow(c, (void **)&b.B, &b.B_cap, (size_t)n, sizeof(long long)) != 0 ||
        rc_grow(c, (void **)&b.flag, &b.flag_cap, 1, sizeof(int)) != 0 ||
        rc_grow(c, (void **)&b.bb, &b.bb_cap, 2, sizeof(unsigned long long)) != 0)
        return -1;
    if (hipMemsetAsync(b.flag, 0, sizeof(int), c->s_fit) != hipSuccess) return -1;
    rk_target_keys_kernel<<<(unsigned)((n + 255) / 256), 256, 0, c->s_fit>>>(r->y64, n, b.keys,
                                                                            b.rows, b.flag);
    if (hipGetLastError() != hipSuccess || segmented_sort(c, n, 1, true) != 0) return -1;
    rk_runs_kernel<true><<<1, RK_THREADS, 0, c->s_fit>>>(b.keys_out, b.rows_out, n, 1, b.start_of,
                                                          b.B, b.bb);
    if (hipGetLastError() != hipSuccess) return -1;
    int bad = 0;
    if (hipMemcpyAsync(&bad, b.flag, sizeof(int), hipMemcpyDeviceToHost, c->s_fit) != hipSuccess ||
        hipMemcpyAsync(b.h_bb, b.bb, 2 * sizeof(unsigned long long), hipMemcpyDeviceToHost,
                       c->s_fit) != hipSuccess ||
        hipStreamSynchronize(c->s_fit) != hipSuccess)
        return -1;
    if (bad) return -1; /* a non-finite target has no ranks (metrics.rs:1267) */
    b.rank_ready = 1;
    return 0;
}

/* The record operators with two children (ft_is_binary's set). */
bool is_binary_code(uint32_t op)
{
    return op == OP_ADD || op == OP_SUB || op == OP_MUL || op == OP_DIV || op == OP_POW;
}

/* The records must be a post-order program the kernels can run without a
   stray read: children before parents, constant slots below pcount, input
   columns below v, at most 96 nodes. */
bool stage_args_ok(const RcCtx *c, const unsigned int *prog, const unsigned int *off,
                   const int *pcount, int nsets, int ntrials, int kmax, const double *c0)
{
    if (!c || !prog || !off || !pcount || !c0 || nsets <= 0 || ntrials <= 0 || kmax <= 0 ||
        kmax > FT_KMAX)
        return false;
    const int nv = c->sets[0].v;
    for (int s = 0; s < nsets; ++s) {
        if (off[s + 1] < off[s]) return false;
        const uint32_t words = off[s + 1] - off[s];
        if (words == 0 || words % 4 != 0 || words / 4 > FT_MAX_NODES) return false;
        if (pcount[s] < 0 || pcount[s] > kmax) return false;
        const unsigned int *nd = prog + off[s];
        for (uint32_t i = 0; i < words / 4; ++i) {
            const uint32_t op = nd[4 * i], k0 = nd[4 * i + 1], k1 = nd[4 * i + 2],
                           slot = nd[4 * i + 3];
            if (op == OP_CONST) {
                if (slot >= (uint32_t)pcount[s]) return false;
            } else if (op == OP_VAR) {
                if ((int)slot < 0 || (int)slot >= nv) return false;
            } else if (k0 >= i || (is_binary_code(op) && k1 >= i)) {
                return false;
            }
        }
    }
    return true;
}

} /* namespace */

int rc_order_invalidate(RcCtx *c)
{
    c->order.rank_ready = 0;
    return 0;
}

void rc_order_free(RcCtx *c)
{
    RcOrderBufs &b = c->order;
    void *ptrs[] = {b.in, b.seg, b.keys, b.keys_out, b.rows, b.rows_out,
                    b.start_of, b.temp, b.val, b.out, b.B, b.flag, b.bb, b.mx, b.part};
    for (void *p : ptrs)
        if (p) (void)hipFree(p);
    b = RcOrderBufs();
}

extern "C" {

float rc_order_stat_score_batch(void *ctx, const unsigned int *prog, const unsigned int *off,
                                const int *pcount, int nsets, int ntrials, int kmax,
                                const double *c0, int what, double *out_value, int *out_status)
{
    RcCtx *c = (RcCtx *)ctx;
    if (!stage_args_ok(c, prog, off, pcount, nsets, ntrials, kmax, c0) || !out_value ||
        !out_status || (what != 0 && what != 1))
        return -1.0f;
    RcRows *r = &c->sets[0];
    const int n = r->n;
    const int nsegs = nsets * ntrials;
    const long long total = (long long)n * (long long)nsegs;
    if (n <= 0 || (long long)nsets * ntrials > 0x7fffffffLL || total > 0x7fffffffLL) return -1.0f;
    if (rc_rows_ensure_f64(c, r) != 0) return -1.0f;
    RcOrderBufs &b = c->order;
    StageInput in;
    stage_sets(c, prog, off, pcount, nsets, &in);
    for (int g = 0; g < nsegs; ++g)
        (in.sets[(size_t)(g / ntrials)].t_m > 0 ? in.fast : in.general).push_back(g);
    const bool sorted = what == 1;
    /* Values and statuses come back in one copy. */
    const size_t ns = (size_t)nsegs, out_bytes = 12 * ns;
    if (stage_inputs(c, prog, off, pcount, nsets, nsegs, kmax, c0, nullptr, nullptr, {}, &in) != 0 ||
        (sorted && segment_offsets(c, nsegs, n) != 0) ||
        sort_buffers(c, total, sorted, false) != 0 ||
        rc_grow(c, (void **)&b.val, &b.val_cap, 2 * ns, sizeof(double)) != 0)
        return -1.0f;
    int *d_status = (int *)(b.val + ns);
    if (hipMemsetAsync(d_status, 0, sizeof(int) * ns, c->s_fit) != hipSuccess) return -1.0f;
    (void)hipEventRecord(c->t0, c->s_fit);
    if (launch_keys(c, false, in, kmax, ntrials, d_status) != 0 ||
        (sorted && segmented_sort(c, total, nsegs, false) != 0))
        return -1.0f;
    if (sorted)
        os_mean_kernel<<<(unsigned)nsegs, 64, 0, c->s_fit>>>(b.keys_out, n, nsegs, b.val, d_status);
    else
        os_select_kernel<<<(unsigned)nsegs, SEL_THREADS, 0, c->s_fit>>>(b.keys, n, nsegs, b.val,
                                                                      d_status);
    if (hipGetLastError() != hipSuccess) return -1.0f;
    (void)hipEventRecord(c->t1, c->s_fit);
    b.h_out.resize(out_bytes);
    if (hipMemcpyAsync(b.h_out.data(), b.val, out_bytes, hipMemcpyDeviceToHost, c->s_fit) !=
            hipSuccess ||
        hipStreamSynchronize(c->s_fit) != hipSuccess)
        return -1.0f;
    memcpy(out_value, b.h_out.data(), sizeof(double) * ns);
    memcpy(out_status, b.h_out.data() + sizeof(double) * ns, sizeof(int) * ns);
    float ms = -1.0f;
    (void)hipEventElapsedTime(&ms, c->t0, c->t1);
    return ms;
}

float rc_rank_score_batch(void *ctx, const unsigned int *prog, const unsigned int *off,
                          const int *pcount, int nsets, int ntrials, int kmax, const double *c0,
                          unsigned long long *out, int *out_status, unsigned long long *out_bb)
{
    RcCtx *c = (RcCtx *)ctx;
    if (!stage_args_ok(c, prog, off, pcount, nsets, ntrials, kmax, c0) || !out || !out_status ||
        !out_bb)
        return -1.0f;
    RcRows *r = &c->sets[0];
    const int n = r->n;
    const int nsegs = nsets * ntrials;
    const long long total = (long long)n * (long long)nsegs;
    if (n <= 1 || (long long)nsets * ntrials > 0x7fffffffLL || total > 0x7fffffffLL) return -1.0f;
    if (rank_prepare(c) != 0) return -1.0f;
    RcOrderBufs &b = c->order;
    StageInput in;
    stage_sets(c, prog, off, pcount, nsets, &in);
    for (int g = 0; g < nsegs; ++g)
        (in.sets[(size_t)(g / ntrials)].t_m > 0 ? in.fast : in.general).push_back(g);
    if (stage_inputs(c, prog, off, pcount, nsets, nsegs, kmax, c0, nullptr, nullptr,
                     std::vector<int>((size_t)nsegs, 0), &in) != 0 ||
        segment_offsets(c, nsegs, n) != 0 || sort_buffers(c, total, true, true) != 0 ||
        rc_grow(c, (void **)&b.out, &b.out_cap, 4 * (size_t)nsegs, sizeof(unsigned long long)) != 0)
        return -1.0f;
    (void)hipEventRecord(c->t0, c->s_fit);
    if (launch_keys(c, true, in, kmax, ntrials, in.flags) != 0 ||
        segmented_sort(c, total, nsegs, true) != 0)
        return -1.0f;
    rk_runs_kernel<false><<<(unsigned)nsegs, RK_THREADS, 0, c->s_fit>>>(
        b.keys_out, b.rows_out, n, nsegs, b.start_of, b.B, b.out);
    if (hipGetLastError() != hipSuccess) return -1.0f;
    (void)hipEventRecord(c->t1, c->s_fit);
    if (hipMemcpyAsync(out, b.out, 4 * sizeof(unsigned long long) * (size_t)nsegs,
                       hipMemcpyDeviceToHost, c->s_fit) != hipSuccess ||
        hipMemcpyAsync(out_status, in.flags, sizeof(int) * (size_t)nsegs, hipMemcpyDeviceToHost,
                       c->s_fit) != hipSuccess ||
        hipStreamSynchronize(c->s_fit) != hipSuccess)
        return -1.0f;
    out_bb[0] = b.h_bb[0];
    out_bb[1] = b.h_bb[1];
    float ms = -1.0f;
    (void)hipEventElapsedTime(&ms, c->t0, c->t1);
    return ms;
}

int rc_rank_debug_b(void *ctx, long long *out)
{
    RcCtx *c = (RcCtx *)ctx;
    if (!c || !out || rank_prepare(c) != 0) return -1;
    if (hipMemcpy(out, c->order.B, sizeof(long long) * (size_t)c->sets[0].n,
                  hipMemcpyDeviceToHost) != hipSuccess)
        return -1;
    return 0;
}

float rc_max_scan_batch(void *ctx, const unsigned int *prog, const unsigned int *off,
                        const int *pcount, int nsets, int ntrials, int kmax, const double *c0,
                        const int *coords, const double *levels, RcMaxOut *out)
{
    RcCtx *c = (RcCtx *)ctx;
    if (!stage_args_ok(c, prog, off, pcount, nsets, ntrials, kmax, c0) || !out) return -1.0f;
    RcRows *r = &c->sets[0];
    const int n = r->n;
    const int nsegs = nsets * ntrials;
    if (n <= 0 || (long long)nsets * ntrials > 0x7fffffffLL ||
        (long long)nsegs * (long long)n > 0x7fffffffLL)
        return -1.0f;
    if (rc_rows_ensure_f64(c, r) != 0) return -1.0f;
    RcOrderBufs &b = c->order;
    StageInput in;
    /* Null coords / levels: the maximum only (coordinate -1, level NaN). */
    std::vector<int> hc((size_t)nsegs, -1);
    std::vector<double> hl((size_t)nsegs, __builtin_nan(""));
    if (coords && levels) {
        hc.assign(coords, coords + nsegs);
        hl.assign(levels, levels + nsegs);
    }
    stage_sets(c, prog, off, pcount, nsets, &in);
    /* The record sweep serves a level where the program fits its stack and
       the constant is one leaf (a sum over several is added in another order
       than the adjoint sweep's), the value stream a plain maximum; the rest is
       marked for the general kernel. */
    std::vector<char> stack((size_t)nsets, 0);
    for (int s = 0; s < nsets; ++s)
        stack[(size_t)s] = n <= OR_MAX_ROWS && off[s] % 4 == 0 &&
                           stack_tree(prog + off[s], in.sets[(size_t)s].m);
    auto one_leaf = [&](int s, int slot) {
        int leaves = 0;
        for (int i = 0; i < in.sets[(size_t)s].m; ++i) {
            const unsigned int *w = prog + off[s] + 4 * i;
            leaves += w[0] == OP_CONST && (int)w[3] == slot;
        }
        return leaves == 1;
    };
    std::vector<int> redo((size_t)nsegs, 0), leveled;
    for (int g = 0; g < nsegs; ++g) {
        const int s = g / ntrials;
        const bool want = pcount[s] > 0 && hc[g] >= 0 && hc[g] < pcount[s] && isfinite(hl[g]) &&
                          hl[g] >= 0.0;
        if (want && stack[(size_t)s] && one_leaf(s, hc[g])) leveled.push_back(g);
        else if (!want && in.sets[(size_t)s].t_m > 0) in.fast.push_back(g);
        else redo[(size_t)g] = 1;
    }
    const int nplain = (int)in.fast.size(), nlevel = (int)leveled.size(), nlist = nplain + nlevel;
    in.fast.insert(in.fast.end(), leveled.begin(), leveled.end());
    int tile_rows = 0;
    const int tiles = or_max_tiles(n, std::max(nlist, 1), &tile_rows);
    if (stage_inputs(c, prog, off, pcount, nsets, nsegs, kmax, c0, hc.data(), hl.data(), redo,
                     &in) != 0 ||
        rc_grow(c, (void **)&b.part, &b.part_cap, (size_t)nlist * (size_t)tiles + 1,
                sizeof(OrMax)) != 0 ||
        rc_grow(c, (void **)&b.mx, &b.mx_cap, (size_t)nsegs, sizeof(RcMaxOut)) != 0)
        return -1.0f;
    OrMax *part = (OrMax *)b.part;
    const OrRows rows = {r->cols64, r->y64, n, r->v};
    (void)hipEventRecord(c->t0, c->s_fit);
    or_launch_max(false, nplain, c->s_fit, in.lists, in.d_sets, in.d_code, in.prog, in.c0, kmax,
                  ntrials, in.coords, in.levels, rows, part, tiles, tile_rows, in.flags);
    or_launch_max(true, nlevel, c->s_fit, in.lists + nplain, in.d_sets, in.d_code, in.prog, in.c0,
                  kmax, ntrials, in.coords, in.levels, rows,
                  part + (size_t)nplain * (size_t)tiles, tiles, tile_rows, in.flags);
    if (nlist > 0)
        mx_finish_kernel<<<(unsigned)nlist, 64, 0, c->s_fit>>>(in.lists, nlist, part, tiles, b.mx);
    mx_scan_kernel<<<(unsigned)nsegs, MX_THREADS, 0, c->s_fit>>>(
        in.prog, in.off, in.pcount, in.c0, kmax, in.coords, in.levels, r->cols64, r->y64, n, nsegs,
        ntrials, in.flags, b.mx);
    if (hipGetLastError() != hipSuccess) return -1.0f;
    (void)hipEventRecord(c->t1, c->s_fit);
    if (hipMemcpyAsync(out, b.mx, sizeof(RcMaxOut) * (size_t)nsegs, hipMemcpyDeviceToHost,
                       c->s_fit) != hipSuccess ||
        hipStreamSynchronize(c->s_fit) != hipSuccess)
        return -1.0f;
    float ms = -1.0f;
    (void)hipEventElapsedTime(&ms, c->t0, c->t1);
    return ms;
}

} /* extern "C" */
