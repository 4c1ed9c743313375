// One low-res pixel's convex upsample: the 9 taps, a sub-pixel on the
// fp32-weight fast path and in double (upsample.hip's comment gives the
// arithmetic and its error bound).  Shared by the upsample kernels and by the
// refiner's fused up-mask head (refiner_conv.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "angmf_ref.h"

namespace bvml {

// The float nearest log2(e) (relative error 1.3e-8).
constexpr float kLog2E = 1.44269504088896340736f;

// Relative error of v_exp_f32 on [-126, 0]: at most 8.484e-8 over every float
// there (measured exhaustively on gfx950).  Below -126 it returns 0 (outputs
// are not denormal), so a tap's weight is off by at most 2^-126 of the
// largest: kFlushAbs * |x_n|, summed over the taps once.
constexpr float kExpRel = 8.5e-8f;
constexpr float kFlushAbs = 1.18e-38f;
// Error of t_n = (m_n - max) * log2e: the fp32 subtraction and product
// round once each (2^-24 |t| apiece) and the float log2 e adds 1.34e-8 |t|;
// 2^(t(1+d)) = 2^t (1 + d t ln 2 + ...), so the weight's relative error from
// the argument is at most ln 2 * 1.33e-7 * |t|.
constexpr float kArgRel = 9.3e-8f;
// Largest per-component error the weights may cause in a normalised output:
// 2 bnd / |v| <= kDirBudget.  The fp32 rsq (relative error <= 9.4e-8 over
// every float, measured), the rounding of |v|^2 to fp32 and the final
// rounding add at most 1.9e-7, so the fast path stays within 7.2e-6 of the
// exact result.
constexpr float kDirBudget = 7.0e-6f;
constexpr float kThrScale = 2.0f / kDirBudget;

// Lanes the fast path accepts: |v|^2 in [kMinN2, kMaxN2] keeps the fp32 rsq
// in its normal range.
constexpr float kMinN2 = 1e-30f;
constexpr float kMaxN2 = 1e30f;

// mode bits
constexpr int kNormalize = 1;
constexpr int kExact = 2;

// The 3x3 replicate-padded neighbourhood of one low-res pixel: x at the 9
// taps (tap n at row y - 1 + n/3, column x - 1 + n%3, clamped) and each tap's
// channel norm in fp32 (used only by the error bound).
template <int C>
struct Taps {
    float v[C][9];
    float nrm[9];
    float flush;  // kFlushAbs * sum of nrm
};

template <int C>
__device__ __forceinline__ void load_taps(const float* __restrict__ xb, long long HW, int H,
                                          int W, int y, int x, Taps<C>& t) {
    const long long row[3] = {(long long)(y > 0 ? y - 1 : 0) * W, (long long)y * W,
                              (long long)(y + 1 < H ? y + 1 : H - 1) * W};
    const int col[3] = {x > 0 ? x - 1 : 0, x, x + 1 < W ? x + 1 : W - 1};
    float q_sum = 0.0f;
#pragma unroll
    for (int n = 0; n < 9; ++n) {
        const long long q = row[n / 3] + col[n % 3];
        float s2 = 0.0f;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            t.v[c][n] = xb[c * HW + q];
            s2 = fmaf(t.v[c][n], t.v[c][n], s2);
        }
        t.nrm[n] = sqrtf(s2);
        q_sum += t.nrm[n];
    }
    t.flush = kFlushAbs * q_sum;
}

// One sub-pixel in double precision: the reference's formula (exp of m - max,
// w = e / sum, sum of w * x, 1 / max(sqrt(|v|^2), eps)) with the library's
// double exp, accumulated as sum(e * x) / sum(e) in one pass over the taps.
template <int C>
__device__ __forceinline__ void exact_subpixel(const float (&m)[9], const Taps<C>& t,
                                               bool normalize, double eps, float (&o)[C]) {
#pragma clang fp contract(off)
    bool nan = false;
#pragma unroll
    for (int n = 0; n < 9; ++n) nan |= __builtin_isnan(m[n]);
    double mx = m[0];
#pragma unroll
    for (int n = 1; n < 9; ++n)
        if ((double)m[n] > mx) mx = m[n];
    double sum = 0.0, v[C];
#pragma unroll
    for (int c = 0; c < C; ++c) v[c] = 0.0;
#pragma unroll
    for (int n = 0; n < 9; ++n) {
        const double e = nan ? __builtin_nan("") : exp((double)m[n] - mx);
        sum += e;
#pragma unroll
        for (int c = 0; c < C; ++c) v[c] += e * (double)t.v[c][n];
    }
    const double rsum = 1.0 / sum;
    double inv = 1.0;
    if (normalize) {
        double n2 = 0.0;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            v[c] *= rsum;
            n2 += v[c] * v[c];
        }
        inv = 1.0 / smax(sqrt(n2), eps);
    } else {
        inv = rsum;
    }
#pragma unroll
    for (int c = 0; c < C; ++c) o[c] = (float)(v[c] * inv);
}

// One sub-pixel on the fp32-weight fast path.  Returns false (o unset) when
// the error bound, a special value or kExact calls for the double body.
// eps_s = 1.01 * eps in float (0 when eps <= 0 or NaN).
template <int C>
__device__ __forceinline__ bool fast_subpixel(const float (&m)[9], const Taps<C>& t, int mode,
                                              float eps_s, float (&o)[C]) {
    float mx = m[0];
#pragma unroll
    for (int n = 1; n < 9; ++n) mx = fmaxf(mx, m[n]);
    double S = 0.0, v[C];
#pragma unroll
    for (int c = 0; c < C; ++c) v[c] = 0.0;
    float bnd = t.flush;
#pragma unroll
    for (int n = 0; n < 9; ++n) {
        const float tn = (m[n] - mx) * kLog2E;
        const float e = __builtin_amdgcn_exp2f(tn);
        const double ed = e;
        S += ed;
#pragma unroll
        for (int c = 0; c < C; ++c) v[c] = fma(ed, (double)t.v[c][n], v[c]);
        bnd = fmaf(e * t.nrm[n], fmaf(-tn, kArgRel, kExpRel), bnd);
    }
    const bool normalize = (mode & kNormalize) != 0;
    bool fast = (mode & kExact) == 0;
    if (normalize) {
        double n2 = 0.0;
#pragma unroll
        for (int c = 0; c < C; ++c) n2 = fma(v[c], v[c], n2);
        const float n2f = (float)n2;
        const float thr = fmaxf(bnd * kThrScale, eps_s * (float)S);
        fast = fast && n2f >= fmaxf(thr * thr, kMinN2) && n2f <= kMaxN2;
        if (fast) {
            const double r = __builtin_amdgcn_rsqf(n2f);
#pragma unroll
            for (int c = 0; c < C; ++c) o[c] = (float)(v[c] * r);
        }
    } else if (fast) {
        const double inv = 1.0 / S;
#pragma unroll
        for (int c = 0; c < C; ++c) o[c] = (float)(v[c] * inv);
    }
    return fast;
}

}  // namespace bvml
