// pf_common.hpp -- helpers shared by host and device code of the particle
// filter library: packed symmetric indexing, the deterministic exp used by the
// resampler, fixed-point weights and the exact systematic thresholds.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cmath>

namespace mkfbt {

// fma(a, b, c) for the deterministic polynomials.  On the device it is the
// three-address v_fma_f64: the compiler's own FP64 FMA selection ties the
// addend to the result register, so a loop-invariant coefficient held in a
// register is copied before every Horner step; this form reads it in place.
// Either way one correctly rounded fused multiply-add, as on the host.
__host__ __device__ inline double dfma(double a, double b, double c)
{
#if defined(__HIP_DEVICE_COMPILE__)
    double r;
    asm("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
#else
    return fma(a, b, c);
#endif
}

typedef unsigned __int128 u128;

// Packed upper-triangular index of (i, j), i <= j, row-major, n x n.
__host__ __device__ constexpr int pk(int n, int i, int j)
{
    return i <= j ? i * n - (i * (i - 1)) / 2 + (j - i) : j * n - (j * (j - 1)) / 2 + (i - j);
}

__host__ __device__ constexpr int npacked(int n) { return n * (n + 1) / 2; }

// exp(x) for x <= 0 from IEEE-exact operations only (rint, fma, ldexp):
// Cody-Waite reduction with the fdlibm split of ln 2 and the degree-12 Taylor
// polynomial on |r| <= ln2/2.  Host and device builds return identical bits,
// which makes the fixed-point resampling weights below reproducible anywhere.
__host__ __device__ inline double det_exp(double x)
{
    if (!(x >= -745.0)) return 0.0;
    if (x > 709.0) x = 709.0;
    const double n = rint(x * 1.4426950408889634074);
    double r = fma(-n, 6.93147180369123816490e-01, x);
    r = fma(-n, 1.90821492927058770002e-10, r);
    double p = 1.0 / 479001600.0;
    p = dfma(p, r, 1.0 / 39916800.0);
    p = dfma(p, r, 1.0 / 3628800.0);
    p = dfma(p, r, 1.0 / 362880.0);
    p = dfma(p, r, 1.0 / 40320.0);
    p = dfma(p, r, 1.0 / 5040.0);
    p = dfma(p, r, 1.0 / 720.0);
    p = dfma(p, r, 1.0 / 120.0);
    p = dfma(p, r, 1.0 / 24.0);
    p = dfma(p, r, 1.0 / 6.0);
    p = dfma(p, r, 0.5);
    p = dfma(p, r, 1.0);
    p = dfma(p, r, 1.0);
    return ldexp(p, (int)n);
}

// v in [0, 1] -> floor(v * 2^32), exactly.
__host__ __device__ inline uint64_t fixed32(double v)
{
    if (!(v > 0.0)) return 0;
    const double t = floor(ldexp(v, 32));
    if (t >= 4294967296.0) return (uint64_t)1 << 32;
    return (uint64_t)(uint32_t)t;
}

// Fixed-point weight of a log-weight relative to the maximum.
__host__ __device__ inline uint64_t qlog(double lw, double lmax)
{
    return (std::isfinite(lw) && std::isfinite(lmax)) ? fixed32(det_exp(lw - lmax)) : 0;
}

// Block-scaled log-weights (the resampler of log-weights).  A block of
// kWeightsBlock consecutive log-weights whose largest finite value is m is
// scaled by 2^-e with e = block_pow(m) = ceil(m log2 e), so that
// q_i = floor(2^32 exp(lw_i - e ln 2)) <= 2^32 and the block's largest q is
// at least 2^31; a block without a finite log-weight has e = kPowEmpty and
// q = 0.  Blocks are aligned by right shifts of E - e, E the largest e, so
// every prefix sum stays an exact integer and no pass over the weights needs
// the global maximum first.
constexpr int kPowEmpty = -2147483647 - 1;
constexpr int kPowLimit = 1 << 30;

__host__ __device__ inline int block_pow(double m)
{
    const double c = ceil(m * 1.4426950408889634);
    return c > (double)kPowLimit ? kPowLimit : (c < -(double)kPowLimit ? -kPowLimit : (int)c);
}

__host__ __device__ inline double pow_ref(int e) { return (double)e * 0.6931471805599453; }

__host__ __device__ inline uint64_t qlog_pow(double lw, int e)
{
    return (std::isfinite(lw) && e != kPowEmpty) ? fixed32(det_exp(lw - pow_ref(e))) : 0;
}

// Right shift aligning a block of exponent e to the largest exponent E (64:
// the block contributes nothing).
__host__ __device__ inline int pow_shift(int E, int e)
{
    if (e == kPowEmpty || E == kPowEmpty) return 64;
    const long long d = (long long)E - (long long)e;
    return d >= 64 ? 64 : (int)d;
}

__host__ __device__ inline uint64_t shr64(uint64_t x, int s) { return s >= 64 ? 0 : x >> s; }

// Systematic resampling of N outputs: output i takes the first input whose
// inclusive prefix C satisfies C N 2^32 > (i 2^32 + U) total, i.e. C > f_i
// with the integer f_i = floor((i 2^32 + U) total / (N 2^32))
//                     = floor((i total + floor(U total / 2^32)) / N).
// With total = qt N + rt and floor(U total / 2^32) = qv N + rv this is
// i qt + qv + floor((i rt + rv) / N): the two divisions by N are made once,
// and the per-output one has a dividend below 2^53 (i, rt < N <= 2^26,
// total <= 2^52), where the product with 1 / N in FP64 is off by at most one.
// The searches then compare 64-bit prefixes with f_i.
__host__ __device__ inline uint64_t div_near(uint64_t s, uint32_t n, double inv, uint64_t &rem)
{
    uint64_t q = (uint64_t)((double)s * inv);
    int64_t r = (int64_t)(s - q * n);
    if (r < 0) {
        --q;
        r += n;
    } else if (r >= (int64_t)n) {
        ++q;
        r -= n;
    }
    rem = (uint64_t)r;
    return q;
}

struct SysThresholds {
    uint64_t qt, qv, rv;
    uint32_t rt, n;
    double inv;
    __host__ __device__ SysThresholds(uint64_t total, uint32_t U, uint32_t N) : n(N), inv(1.0 / (double)N)
    {
        uint64_t r;
        qt = div_near(total, n, inv, r);
        rt = (uint32_t)r;
        qv = div_near((uint64_t)(((u128)total * U) >> 32), n, inv, rv);
    }
    // f_i for i < N
    __host__ __device__ uint64_t operator()(uint32_t i) const
    {
        const uint64_t s = (uint64_t)i * rt + rv;
        uint32_t q = (uint32_t)((double)s * inv);
        const int64_t r = (int64_t)(s - (uint64_t)q * n);
        q += r < 0 ? -1 : (r >= (int64_t)n ? 1 : 0);
        return qt * i + qv + q;
    }
};

// Component draw resample(gmm.weight, N) as 64-bit keys.  With the cumulative
// fixed-point weights C_k, total T = C_{K-1}, output j draws the first k with
// C_k N 2^32 > (j 2^32 + U) T.  Write C_k N = I T + r (0 <= r < T): since
// j 2^32 + U is an integer, C_k N 2^32 <= (j 2^32 + U) T exactly when
// I 2^32 + ceil(r 2^32 / T) <= j 2^32 + U.  The left side depends on the model
// alone, so the draw compares 64-bit integers.
__host__ inline uint64_t component_key(uint64_t cum, uint64_t total, uint64_t n)
{
    const u128 x = (u128)cum * n;
    const u128 whole = x / total, rest = x % total;
    return (uint64_t)((whole << 32) + ((rest << 32) + total - 1) / total);
}

// Model image of the step kernels: [component keys, K 64-bit words][H
// (m x D), BH (m), R 2x2 blocks (3J), padded to even][per joint the FP64
// innovation block (bh0, bh1, r00, r01, r11) as doubles (5J)], padded to 4
// floats, then [component rows, K x (2 + D + D(D+1)/2)].  Offset of the FP64
// blocks (8-byte aligned) and floats of the part before the component rows:
__host__ __device__ constexpr int image_j64_floats(int K, int m, int D, int J)
{
    return 2 * K + ((m * D + m + 3 * J + 1) & ~1);
}
__host__ __device__ constexpr int image_head_floats(int K, int m, int D, int J)
{
    return (image_j64_floats(K, m, D, J) + 10 * J + 3) & ~3;
}

// A 2 x 2 innovation covariance S = [[s00, s01], [s01, s11]] whose FP32
// Cholesky is not trusted: a pivot that is not positive, or
// det S <= 1e-6 (tr S)^2, i.e. cond(S) >= ~1e6 (for a 2 x 2 SPD matrix
// det / tr^2 = c / (1 + c)^2 with c = 1 / cond).  Such joints are factored in FP64.
__host__ __device__ inline bool innovation_ill(float s00, float s01, float s11)
{
    const float tr = s00 + s11;
    const float det = fmaf(s00, s11, -s01 * s01);
    return !(s00 > 0.f) || !(det > 1e-6f * tr * tr);
}

// Status bits of the device work (FrameScratch::status and the batched
// engine's per-sequence status): the uniform resampling fallback (no positive
// weight), a joint factored in FP64, a joint whose innovation covariance is
// not positive definite even in FP64 (the particle's weight is zero).
constexpr unsigned kStatusDegenerate = 1u;
constexpr unsigned kStatusIllCond = 2u;
constexpr unsigned kStatusNotSpd = 4u;
// LDS budget of the staged image: above it only the head is staged and the
// component rows are read from global memory.
constexpr int kImageLdsBytes = 48 * 1024;

}  // namespace mkfbt
