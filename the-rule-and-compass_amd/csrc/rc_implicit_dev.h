/*
 * Device definitions that the implicit arm's kernels share (rc_implicit.hip,
 * rc_implicit_kern.hip): work items, the operators' values, the zero rule.
 */
#ifndef RC_IMPLICIT_DEV_H
#define RC_IMPLICIT_DEV_H

#include "rc_device.h"

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

constexpr int IM_MAX_NODES = 96;
constexpr int IM_KMAX = 20;
constexpr int IM_STATS = (IM_KMAX + 1) * (IM_KMAX + 2) / 2; /* [J | r] lower triangle */
constexpr int IM_SUMS = 2; /* a score's sums: weighted distances, weights */
constexpr double IM_INV_SQRT_PI = 0.5641895835477563;

enum { IM_SCORE = 0, IM_RSS = 1, IM_JAC = 2 };

struct ImCand {
    uint32_t off; /* first record word */
    int m;        /* nodes */
    int k;        /* constants */
    int fast;     /* 2: runs the four-wide sweep (im_wide_kernel), 1: the
                     register-stack sweep (im_fast_kernel), 0: node arrays */
    int sub;      /* rows of a sub-tile, items of a group (RcSplit) */
    int group;
};

/* The register-stack sweep's limits: values below the top of the stack
   (the post-order evaluation's depth less one) and input columns. */
constexpr int IM_SDEPTH = 8;
constexpr int IM_NVMAX = 4;
/* A stack file: two components of the 8 stack entries, one in elements
   0..7 and one in 8..15 (a 16-element vector is indexed with one register
   move per access; shorter ones are lowered to select chains). */
typedef double im_d16 __attribute__((ext_vector_type(16)));
typedef double im_d4 __attribute__((ext_vector_type(4)));

struct ImItem {
    int cand;
    int row0;
    int rows;
    int pad;
};

/* value_of (fit.rs:1211-1365) for the fit operator set. */
__device__ __forceinline__ double im_value(uint32_t op, double a, double b)
{
    switch (op) {
        case OP_ADD: return a + b;
        case OP_SUB: return a - b;
        case OP_MUL: return a * b;
        case OP_DIV: return fabs(b) < 1e-12 ? RC_F64_NAN : a / b;
        case OP_POW: return pow(a, b);
        case OP_NEG: return -a;
        case OP_EXP: return a > 700.0 ? __builtin_inf() : exp(a);
        case OP_LOG: return log(a);
        case OP_ABS: return fabs(a);
        case OP_SQRT: return sqrt(a);
        case OP_SIN: return sin(a);
        case OP_COS: return cos(a);
        case OP_TAN: return tan(a);
        case OP_SINH: return sinh(a);
        case OP_COSH: return cosh(a);
        case OP_TANH: return tanh(a);
        case OP_SIG: return 1.0 / (1.0 + exp(-a));
        case OP_GAUSS: return exp(-a * a);
        case OP_SQUARE: return a * a;
        case OP_CUBE: return a * a * a;
        case OP_ERF: return erf(a);
        case OP_ERFC: return erfc(a);
        default: return RC_F64_NAN;
    }
}

__device__ __forceinline__ bool im_is_bin(uint32_t op)
{
    return op == OP_ADD || op == OP_SUB || op == OP_MUL || op == OP_DIV || op == OP_POW;
}

/* A local partial's product with a tangent under the adjoint sweep's zero rule
   (a zero adjoint skips its node), and a quotient. */
__device__ __forceinline__ double im_lm(double p, double t)
{
    return (p == 0.0 || t == 0.0) ? 0.0 : p * t;
}
__device__ __forceinline__ double im_ld(double t, double x) { return t == 0.0 ? 0.0 : t / x; }

/* The four-wide sweep's limits: values below the top of the stack and input
   columns. */
constexpr int IM_WDEPTH = 4;
constexpr int IM_WNV = 3;

/* im_pass_kernel for the candidates marked 2, MODE IM_SCORE, IM_RSS or IM_JAC. */
void im_launch_wide(int mode, int nv, int ni, hipStream_t s, const ImItem *items,
                    const ImCand *cands, const uint32_t *rec, const double *cs, int kmax,
                    const double *cols64, const double *w64, int n, int metric, double *part,
                    int pstride, int *bad, const int *run);

#endif
