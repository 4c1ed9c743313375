// The native refiner's own kernels: its ConvGRU's 5x5 and its heads' 3x3
// convolutions (stride 1, zero "same" padding) with everything around them
// fused (src/dsine_refine.cpp:119-159), and the first steps of a forward.
//
// The convolutions are implicit GEMMs on the f16 matrix cores at fp32
// precision.  Every operand, scaled by a power of two to below 2^15, is the
// sum of two halfs, hi = half(v) and lo = half(v - hi); a product is three
// matrix-core products (hi hi + hi lo + lo hi; the omitted lo lo is at most
// 2^-22 of it) summed in fp32.  A value is off by at most 2^-23 of itself down
// to 2^-16 of its scale's bound, below that by at most 2^-39 of the bound.  The
// scales come off the sums exactly.  The weights are split when they are
// packed, each output channel scaled to its largest weight; a map is split by
// the kernel that writes it, by one scale: that of its largest value (of the
// hidden state: the largest of 1 and the decoder's |hidden|, which a ConvGRU
// state never exceeds), but no larger than leaves the sums as precise as the
// activations they go to can use (kBudget).  A value beyond that scale, an
// infinity or a NaN makes the sums of the windows that hold it infinite or NaN,
// and the workgroups that find such sums convolve the fp32 maps on the fp32
// matrix cores instead, as all do whose weights have an infinity or a NaN.
//
// Three v_mfma_f32_16x16x32_f16 (16 cycles each) do the work of eight
// v_mfma_f32_16x16x4_f32 (32 cycles each), and the sums' chains are shorter
// (150 additions instead of 400 for 64 channels and 25 taps): relative rms
// error 4.4e-7 against 7.1e-7 for the fp32 kernel on the same operands.

#include <hip/hip_runtime.h>

#include <climits>
#include <cstdint>

#include "angmf_ref.h"
#include "refiner_kernels.h"
#include "upsample_px.h"

namespace {

using namespace bvml_refine;

typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));

constexpr int kTW = 16;  // tile width: one MFMA column block per tile row

enum Epi : int { kPlain = 0, kGates = 1, kUpdate = 2, kHeads = 3, kUp = 4 };

// A head's small operands in LDS, in words: the three layers' exponents and
// biases, [e0 64][b0 64][e2 64][b2 64][e4 outs][b4 outs], outs rounded up to
// 16; the heads' outputs are at most 64, the up-mask head's 9 taps x 64.
constexpr int kSubs = 64, kUpOuts = 9 * kSubs;
constexpr int head_outs(int epi) { return epi == kUp ? kUpOuts : 64; }
constexpr int head_words(int epi) { return 256 + 2 * head_outs(epi); }

struct KArgs {
    ConvArgs c;
    int wblocks, tiles_x, mgroups;
    uint32_t HW;
};

__device__ __forceinline__ float relu(float v) { return v < 0.0f ? 0.0f : v; }
__device__ __forceinline__ float sigmoid(float x) { return 1.0f / (1.0f + expf(-x)); }
__device__ __forceinline__ float gru_mix(float z, float h, float q) {
#pragma clang fp contract(off)
    const float omz = 1.0f - z;
    return omz * h + z * q;
}
__device__ __forceinline__ uint32_t absbits(float v) {
    return __builtin_bit_cast(uint32_t, v) & 0x7fffffffu;
}
__device__ __forceinline__ uint32_t umax(uint32_t a, uint32_t b) { return a > b ? a : b; }
__device__ __forceinline__ uint32_t wave_max(uint32_t m) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) m = umax(m, (uint32_t)__shfl_xor((int)m, d));
    return m;
}

constexpr uint32_t kInfBits = 0x7f800000u;

// Where a map's scale ends: its bound, times the largest weight of the layers
// that read it, is at most 2^(kBudget + 1).  A value below the bound is off by at
// most 2^-40 of it, so a sum of 1,650 products with weights spread up to the
// largest by about 2^-40 2^11 sqrt(1650) / 3 = 2^-25 (rms): the rounding of a
// gate of unit scale, a tenth of what an fp32 sum of so many terms is off.
// Features up to 2^16 fit beside weights of the usual +-1/sqrt(fan_in), up to
// 2^9 beside a weight of 2.
constexpr int kBudget = 10;
// The bits of the largest power of two that times wmax (finite) stays below
// 2^(budget + 1), at most 2^64.
__device__ __forceinline__ uint32_t limit_bits(uint32_t wmax, int budget) {
    const int e = 2 * 127 + budget - (int)(wmax >> 23);  // (at least `budget`)
    return (uint32_t)(e < 191 ? e : 191) << 23;
}
// The same for a pixel's activations, which its largest one scales, and the 64
// inputs of a 1x1 layer: the sums are off by 2^-40 2^11 sqrt(64) / 3 = 2^-27.6.
// From the limit on, and at an infinity or a NaN, a row takes fp32 products.
constexpr int kHeadBudget = 10;
__device__ __forceinline__ uint32_t head_limit(uint32_t wmax) {
    return wmax < kInfBits ? limit_bits(wmax, kHeadBudget) : 0u;
}

// The power of two that brings a magnitude of these bits into [2^14, 2^15),
// as its exponent (at most 126, so that it is a normal float: a magnitude
// below 2^-112 stays smaller).
__device__ __forceinline__ int scale_exp(uint32_t bits) {
    const int n = 14 + 127 - (int)(bits >> 23);
    return n < 126 ? n : 126;
}
__device__ __forceinline__ float pow2(int n) {
    return __builtin_bit_cast(float, (uint32_t)(n + 127) << 23);
}

template <int N, typename H>
__device__ __forceinline__ void split_to(const float (&v)[N], H& hi, H& lo) {  // already scaled
#pragma unroll
    for (int j = 0; j < N; ++j) {
        hi[j] = (_Float16)v[j];
        lo[j] = (_Float16)(v[j] - (float)hi[j]);
    }
}

// Raw buffer loads of packed weights: the descriptor in scalar registers, a
// per-lane byte offset and a wave-uniform one.
constexpr int kBufferWord3 = 0x00020000;  // gfx9 raw-buffer descriptor word 3
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_of(const float* w, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(w), (short)0, (int)bytes,
                                             kBufferWord3);
}
__device__ __forceinline__ h8 ld16(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t soff) {
    return __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, (int)soff, 0));
}

// K: kernel size; TAIL: the two extra channels; each wave MB 16-channel
// blocks x NB tile rows; WM x WN waves along the channels and the rows; KS
// groups of those waves that split the reduction's steps; AD: steps whose
// weights are in flight.
template <int K_, bool TAIL_, int MB_, int NB_, int WM_, int WN_, int KS_, int AD_, int EPI_>
struct Shape {
    static constexpr int K = K_, MB = MB_, NB = NB_, WM = WM_, WN = WN_, KS = KS_, AD = AD_,
                         EPI = EPI_;
    static constexpr bool TAIL = TAIL_;
    // registers for two waves on a SIMD, or (the up-mask head, with 9 blocks of
    // weights resident) one: two spilled 430 bytes a lane
    static constexpr int kWavesPerSimd = EPI == kUp ? 1 : 2;
    static constexpr int kWaves = WM * WN * KS, kThreads = 64 * kWaves;
    static constexpr int TH = NB * WN;
    static constexpr int HR = TH + K - 1, HC = kTW + K - 1, HS = HR * HC;
    // a multiple of 16 pixels: 256 bytes, so the four channel groups that a B
    // read takes fall on the banks its 16 columns leave free
    static constexpr int HSP = (HS + 15) / 16 * 16;
    static constexpr int kHaloBytes = 2 * 8 * HSP * 16;
    static constexpr int kTailPx = HS + 8;
    static constexpr int kTailBytes = TAIL ? 2 * kTailPx * 4 : 0;
    // the groups' partial sums, all but each group's own columns
    static constexpr int kXchBytes = KS > 1 ? WM * WN * (KS - 1) * MB * NB * 1024 : 0;
    // the up-mask head's activations, their exponents, each row's flag
    static constexpr int kFragBytes = EPI == kUp ? TH * (4096 + 64 + 16) : 0;
    static constexpr int kMainBytes = kHaloBytes + kTailBytes;
    static constexpr int kShared1 = kMainBytes > kXchBytes ? kMainBytes : kXchBytes;
    static constexpr int kParamAt = ((kShared1 > kFragBytes ? kShared1 : kFragBytes) + 15) / 16 * 16;
    static constexpr int kParamBytes = EPI >= kHeads ? WM * head_words(EPI) * 4 : 0;
    // the up-mask head's normals, with a border of one pixel
    static constexpr int kPredAt = kParamAt + kParamBytes;
    static constexpr int kPredBytes = EPI == kUp ? (TH + 2) * (kTW + 2) * 16 : 0;
    static constexpr int kRedoAt = kPredAt + kPredBytes;
    static constexpr int kLdsBytes = kRedoAt + 16;
    static constexpr int NC = NB >= KS ? NB / KS : 1;  // columns (tile rows) a wave finishes
    static_assert(NB % KS == 0 || NB < KS, "whole columns per group");
    static_assert(AD % 2 == 0, "B operands alternate between two slots");
};

// Workgroup bx of nbx of one convolution.
template <class S>
__device__ __forceinline__ void conv_group(const KArgs& a, int bx, int nbx, char* lds) {
    constexpr int K = S::K, P = K / 2, TAPS = K * K, MAIN = 2 * TAPS;
    constexpr bool TAIL = S::TAIL;
    constexpr int STEPS = split_steps(K, TAIL);
    constexpr int MB = S::MB, NB = S::NB, WM = S::WM, WN = S::WN, KS = S::KS, AD = S::AD;
    constexpr int HC = S::HC, HS = S::HS, HSP = S::HSP, NC = S::NC, EPI = S::EPI;

    const ConvArgs& c = a.c;
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, col = lane & 15;
    const int wm = wave % WM, wn = (wave / WM) % WN, ks = wave / (WM * WN);
    // each XCD takes a contiguous run of (tile, channel group) pairs
    // (workgroups go to the 8 XCDs in turn), so neighbouring tiles share
    // their halo lines in one L2
    const int xcd = bx & 7;
    const int id = xcd * (nbx >> 3) + (xcd < (nbx & 7) ? xcd : (nbx & 7)) + (bx >> 3);
    const int tile = id / a.mgroups, mg = id - tile * a.mgroups;
    const int tx0 = (tile % a.tiles_x) * kTW, ty0 = (tile / a.tiles_x) * S::TH;
    const int mb0 = (EPI == kUp ? 12 : mg * (MB * WM)) + MB * wm;  // the wave's first M-block
    const int H = c.H, W = c.W;
    const size_t HW = a.HW;

    // the wave's steps of the reduction
    const int st0 = KS > 1 ? STEPS * ks / KS : 0;
    const int st1 = KS > 1 ? STEPS * (ks + 1) / KS : STEPS;
    const int sm1 = st1 < MAIN ? st1 : MAIN;  // (the tail's steps come last)

    const int* const wexp = reinterpret_cast<const int*>(c.wp);
    const uint32_t whead = split_head_words(a.wblocks);
    const Info* const info = reinterpret_cast<const Info*>(c.info);

    const __amdgpu_buffer_rsrc_t wr = rsrc_of(c.wp + whead, (uint32_t)a.wblocks * STEPS * 2048u);
    const uint32_t lane16 = 16u * (uint32_t)lane;
    h8 aw[AD][MB][2];
    auto a_load = [&](int st, int slot) {
#pragma unroll
        for (int m = 0; m < MB; ++m) {
            const uint32_t so = ((uint32_t)(mb0 + m) * STEPS + (uint32_t)st) * 2048u;
            aw[slot][m][0] = ld16(wr, lane16, so);
            aw[slot][m][1] = ld16(wr, lane16 + 1024u, so);
        }
    };

    constexpr bool HEAD = EPI == kHeads || EPI == kUp;
    constexpr int OUTS = head_outs(EPI);

    // lane (g, col), register r of a block's sums is output channel
    // 16 (mb0 + m) + 4 g + r (in the packed order) at pixel (row(j), tx0 + col)
    const int x = tx0 + col;
    auto row_of = [&](int j) { return ty0 + wn * NB + j * KS + ks; };
    // channels 16 q + 4 g .. + 3 of a pixel, in c4
    auto c4_at = [&](int q, uint32_t px) { return ((size_t)(4 * q + g) * HW + px) * 4; };
    // what the gates' and the update's epilogues read, fetched before the sums
    // where the reduction is split (few rows a wave, small grids), else after
    constexpr bool EARLY = KS > 1 && (EPI == kGates || EPI == kUpdate);
    constexpr int NE = EPI == kGates ? MB / 2 : EPI == kUpdate ? MB : 1;
    v4f ep[3][NC][NE], eb[2][NE];
    auto epilogue_loads = [&]() {
        const int xc = x < W ? x : W - 1, q0 = EPI == kGates ? mb0 / 2 : mb0;
#pragma unroll
        for (int p = 0; p < NE; ++p) {
            eb[0][p] = *reinterpret_cast<const v4f*>(c.b0 + 16 * (q0 + p) + 4 * g);
            if (EPI == kGates)
                eb[1][p] = *reinterpret_cast<const v4f*>(c.b1 + 16 * (q0 + p) + 4 * g);
#pragma unroll
            for (int j = 0; j < NC; ++j) {
                const int y = row_of(j) < H ? row_of(j) : H - 1;
                const uint32_t px = (uint32_t)(y * W + xc);
                const size_t at = c4_at(q0 + p, px);
                if (EPI == kGates) {
                    ep[0][j][p] = *reinterpret_cast<const v4f*>(c.s0 + c4_at(mb0 + 2 * p, px));
                    ep[1][j][p] = *reinterpret_cast<const v4f*>(c.s0 + c4_at(mb0 + 2 * p + 1, px));
                } else {
                    ep[0][j][p] = *reinterpret_cast<const v4f*>(c.s0 + at);
                    ep[1][j][p] = *reinterpret_cast<const v4f*>(c.z + at);
                }
                ep[2][j][p] = *reinterpret_cast<const v4f*>(c.hf + at);
            }
        }
    };

    v4f acc[MB][NB];
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int n = 0; n < NB; ++n) acc[m][n] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

    // Everything the sums start from goes out before anything is waited for:
    // one memory latency, where a grid is too small to hide several (whatever
    // the scales turn out to be: the split map is allocated, if not written).
    // the halo to LDS with direct-to-LDS loads, 16 bytes a lane: the waves
    // share the 16 planes (hi, lo x channel group)
    const char* const xs = static_cast<const char*>(c.xs);
    constexpr int PPW = (16 + S::kWaves - 1) / S::kWaves;
    const int pl0 = wave * PPW, pl1 = pl0 + PPW < 16 ? pl0 + PPW : 16;
#pragma unroll
    for (int ch = 0; ch < (HS + 63) / 64; ++ch) {
        const int px = ch * 64 + lane;
        const int y = ty0 + px / HC - P, x = tx0 + px % HC - P;
        if (px < HS) {
            if (y >= 0 && y < H && x >= 0 && x < W) {
                const char* src = xs + ((size_t)pl0 * HW + (uint32_t)(y * W + x)) * 16;
#pragma unroll
                for (int p = 0; p < PPW; ++p)
                    if (16 % S::kWaves == 0 || pl0 + p < pl1) __builtin_amdgcn_global_load_lds(
                        static_cast<const void*>(src + (size_t)p * HW * 16),
                        reinterpret_cast<__attribute__((address_space(3))) void*>(
                            reinterpret_cast<uintptr_t>(
                                lds + ((pl0 + p) * HSP + ch * 64) * 16)),
                        16, 0, 0);
            } else {
#pragma unroll
                for (int p = 0; p < PPW; ++p)
                    if (16 % S::kWaves == 0 || pl0 + p < pl1)
                        *reinterpret_cast<v4u*>(lds + ((pl0 + p) * HSP + px) * 16) =
                            v4u{0, 0, 0, 0};
            }
        }
    }
    // the first steps' weights, in flight beside the halo
#pragma unroll
    for (int u = 0; u < AD; ++u) a_load(st0 + u < st1 ? st0 + u : st1 - 1, u);
    uint32_t* const tl = reinterpret_cast<uint32_t*>(lds + S::kHaloBytes);
    if constexpr (TAIL) {
#pragma unroll
        for (int i = 0; i < (S::kTailPx + S::kThreads - 1) / S::kThreads; ++i) {
            const int px = tid + i * S::kThreads;
            const int y = ty0 + px / HC - P, x = tx0 + px % HC - P;
            const bool in = px < HS && y >= 0 && y < H && x >= 0 && x < W;
            const uint32_t at = in ? (uint32_t)(y * W + x) : 0u;
            const uint32_t hi = c.tail[at], lo = c.tail[HW + at];
            if (px < S::kTailPx) {
                tl[px] = in ? hi : 0u;
                tl[S::kTailPx + px] = in ? lo : 0u;
            }
        }
    }
    // the heads' small operands, for the layers after the sums
    if constexpr (HEAD) {
        static_assert(!HEAD || MB == 4, "one head per wave");
        for (int h = 0; h < WM; ++h) {
            const int hd = EPI == kUp ? 3 : mg * WM + h;
            const int nout = c.nout[hd];
            const int* const e2 = reinterpret_cast<const int*>(c.w2[hd]);
            const int* const e4 = reinterpret_cast<const int*>(c.w4[hd]);
            int* const pe = reinterpret_cast<int*>(lds + S::kParamAt) + h * head_words(EPI);
            float* const pb = reinterpret_cast<float*>(pe);
            for (int i = tid; i < 64; i += S::kThreads) {
                pe[i] = wexp[64 * hd + i];
                pb[64 + i] = c.hb0[hd][i];
                pe[128 + i] = e2[i];
                pb[192 + i] = c.hb2[hd][i];
            }
            for (int i = tid; i < OUTS; i += S::kThreads) {
                pe[256 + i] = i < (nout + 15) / 16 * 16 ? e4[i] : 0;
                pb[256 + OUTS + i] = i < nout ? c.b4[hd][i] : 0.0f;
            }
        }
    }
    if constexpr (EPI == kUp) {
        // each pixel's normal and its length (bvml::load_taps's)
        for (int i = tid; i < (S::TH + 2) * (kTW + 2); i += S::kThreads) {
            int y = ty0 + i / (kTW + 2) - 1, x = tx0 + i % (kTW + 2) - 1;
            y = y < 0 ? 0 : y < H ? y : H - 1;
            x = x < 0 ? 0 : x < W ? x : W - 1;
            v4f v;
            float s2 = 0.0f;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                v[k] = c.pred[k * HW + (uint32_t)(y * W + x)];
                s2 = fmaf(v[k], v[k], s2);
            }
            v[3] = sqrtf(s2);
            reinterpret_cast<v4f*>(lds + S::kPredAt)[i] = v;
        }
    }

    if constexpr (EARLY) epilogue_loads();
    const int xn = info->n[c.which];
    const bool wide = info->wide[c.which] != 0;
    bool exact = (uint32_t)wexp[16 * a.wblocks] >= kInfBits;  // fp32 products
    int* const redo = reinterpret_cast<int*>(lds + S::kRedoAt);
    if (KS > 1 && tid == 0) *redo = exact;
    __builtin_amdgcn_s_waitcnt(0);  // the direct-to-LDS loads
    __syncthreads();

    if (__builtin_expect(!exact, 1)) {
        const char* const hb = lds + (g * HSP + wn * NB * HC + col) * 16;
        h8 bw[2][NB][2];
        auto b_load = [&](int st, int slot) {
            const int cc = st >= TAPS ? 1 : 0, tap = st - cc * TAPS;
            const int off = (cc * 4 * HSP + (tap / K) * HC + tap % K) * 16;
            const char* p = hb + off;
#pragma unroll
            for (int n = 0; n < NB; ++n) {
                bw[slot][n][0] = *reinterpret_cast<const h8*>(p + n * HC * 16);
                bw[slot][n][1] = *reinterpret_cast<const h8*>(p + (8 * HSP + n * HC) * 16);
            }
        };
        auto products = [&](int as, int bs) {
#pragma unroll
            for (int p = 0; p < 3; ++p)
#pragma unroll
                for (int m = 0; m < MB; ++m)
#pragma unroll
                    for (int n = 0; n < NB; ++n)
                        acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                            aw[as][m][p == 0 ? 1 : 0], bw[bs][n][p == 1 ? 1 : 0], acc[m][n], 0, 0,
                            0);
        };
        int st = st0;
        b_load(st < MAIN ? st : MAIN - 1, 0);
        for (; st + AD <= sm1; st += AD) {
#pragma unroll
            for (int u = 0; u < AD; ++u) {
                const int nx = st + u + 1;
                b_load(nx < MAIN ? nx : MAIN - 1, (u + 1) & 1);
                __builtin_amdgcn_sched_barrier(0);
                products(u, u & 1);
                const int na = st + u + AD;
                a_load(na < st1 ? na : st1 - 1, u);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // the steps left (their weights are in the slots from 0 on)
#pragma unroll
        for (int u = 0; u < AD - 1; ++u) {
            if (st + u < sm1) {
                const int nx = st + u + 1;
                b_load(nx < MAIN ? nx : MAIN - 1, (u + 1) & 1);
                products(u, u & 1);
            }
        }
        if constexpr (TAIL) {
            // K = 5: two rows of 8 taps per step (5 of them real), K = 3: the
            // rows of 4 taps (3 real), both channels of a tap together; a
            // lane's 8 values are 4 taps of one row, at 4 pixels of the tail
            for (int ts = st0 > MAIN ? st0 : MAIN; ts < st1; ++ts) {
                a_load(ts, 0);
                const int t = ts - MAIN;
                int row = K == 5 ? 2 * t + (g >> 1) : g;
                row = row < K ? row : K - 1;  // (zero weights there)
                const int kx = K == 5 ? 4 * (g & 1) : 0;
                const int at = (wn * NB + row) * HC + col + kx;
#pragma unroll
                for (int n = 0; n < NB; ++n) {
                    v4u hi, lo;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        hi[q] = tl[at + n * HC + q];
                        lo[q] = tl[S::kTailPx + at + n * HC + q];
                    }
                    bw[0][n][0] = __builtin_bit_cast(h8, hi);
                    bw[0][n][1] = __builtin_bit_cast(h8, lo);
                }
                products(0, 0);
            }
        }
        // a window holds a value beyond the scale, an infinity or a NaN
        if (__builtin_expect(wide, 0)) {
            bool bad = false;
#pragma unroll
            for (int m = 0; m < MB; ++m)
#pragma unroll
                for (int n = 0; n < NB; ++n)
#pragma unroll
                    for (int r = 0; r < 4; ++r) bad |= absbits(acc[m][n][r]) >= kInfBits;
            exact = __any(bad);
            if (KS > 1 && exact && lane == 0) *redo = 1;
        }
    }

    if constexpr (KS > 1) {
        __syncthreads();  // every wave is done with the halo
        // (the waves that split the reduction decide together)
        if (__builtin_expect(wide, 0)) exact = __builtin_amdgcn_readfirstlane(*redo) != 0;
    }
    if (__builtin_expect(exact, 0)) {
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
            for (int n = 0; n < NB; ++n) acc[m][n] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
        // fp32 products of the fp32 map and the unsplit weights: one 16x16x4
        // step per tap and 4 channels.  A row of taps is in flight through the
        // products of the one before it (each step waiting for its own loads took
        // a forward with one infinite hidden value at 256 x 256 to 3863 us, so
        // 2573).  (Buffer loads: 0 beyond the map, by their offset.)
        constexpr int GROUPS = split_groups(TAIL), ROWS = 16 / KS * K;
        const __amdgpu_buffer_rsrc_t rw = rsrc_of(
            c.wp + whead + (size_t)a.wblocks * STEPS * 512,
            (uint32_t)a.wblocks * TAPS * GROUPS * 256u);
        const __amdgpu_buffer_rsrc_t rx = rsrc_of(c.x32, 256u * a.HW);
        float af[2][K][MB], bf[2][K][NB];
        auto row_load = [&](__amdgpu_buffer_rsrc_t rm, uint32_t px_bytes, uint32_t base, bool use,
                            int cg, int ky, int slot) {
#pragma unroll
            for (int kx = 0; kx < K; ++kx) {
#pragma unroll
                for (int m = 0; m < MB; ++m)
                    af[slot][kx][m] = __builtin_bit_cast(
                        float, __builtin_amdgcn_raw_buffer_load_b32(
                                   rw, 4 * lane,
                                   (((mb0 + m) * GROUPS + cg) * TAPS + ky * K + kx) * 256, 0));
                const int x = tx0 + col + kx - P;
#pragma unroll
                for (int n = 0; n < NB; ++n) {
                    const int y = ty0 + wn * NB + n + ky - P;
                    const bool in = use && y >= 0 && y < H && x >= 0 && x < W;
                    const uint32_t at = base + px_bytes * (uint32_t)(y * W + x);
                    bf[slot][kx][n] = __builtin_bit_cast(
                        float, __builtin_amdgcn_raw_buffer_load_b32(
                                   rm, (int)(in ? at : 0xf0000000u), 0, 0));
                }
            }
        };
        auto row_products = [&](int slot) {
#pragma unroll
            for (int kx = 0; kx < K; ++kx)
#pragma unroll
                for (int m = 0; m < MB; ++m)
#pragma unroll
                    for (int n = 0; n < NB; ++n)
                        acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                            af[slot][kx][m], bf[slot][kx][n], acc[m][n], 0, 0, 0);
        };
        auto load = [&](int i, int slot) {
            i = i < ROWS ? i : ROWS - 1;
            const int cg = ks + i / K * KS;
            // channel 4 cg + g: NCHW in the context's map, c4 in the others'
            const uint32_t base = EPI == kPlain ? 4u * (4 * cg + g) * a.HW : 16u * cg * a.HW + 4 * g;
            row_load(rx, EPI == kPlain ? 4 : 16, base, true, cg, i % K, slot);
        };
        static_assert(ROWS % 2 == 0, "two rows a round");
        load(0, 0);
        for (int i = 0; i < ROWS; i += 2) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                load(i + u + 1, (u + 1) & 1);
                __builtin_amdgcn_sched_barrier(0);
                row_products(u);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if constexpr (TAIL) {
            const __amdgpu_buffer_rsrc_t ru = rsrc_of(c.uv, 8u * a.HW);
            if (ks == 0)
                for (int ky = 0; ky < K; ++ky) {
                    row_load(ru, 4, 4u * g * a.HW, g < 2, 16, ky, 0);
                    row_products(0);
                }
        }
    }
    // the heads' second layer's weights, in flight through what follows
    constexpr uint32_t kHead64 = split1x1_head_words(64);
    h8 w2v[HEAD ? 4 : 1][2][2];
    auto w_load = [&](__amdgpu_buffer_rsrc_t rr, int ob, h8 (&w)[2][2]) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            w[q][0] = ld16(rr, lane16, (uint32_t)(ob * 2 + q) * 2048u);
            w[q][1] = ld16(rr, lane16 + 1024u, (uint32_t)(ob * 2 + q) * 2048u);
        }
    };
    const int hd = EPI == kUp ? 3 : HEAD ? mg * WM + wm : 0;
    if constexpr (HEAD) {
        const __amdgpu_buffer_rsrc_t r2 = rsrc_of(c.w2[hd] + kHead64, 4 * 2 * 2048u);
#pragma unroll
        for (int mo = 0; mo < 4; ++mo) w_load(r2, mo, w2v[mo]);
    }

    // the groups' partial sums meet: group ks finishes columns n = ks, ks + KS, ...
    v4f own[MB][NC];
    if constexpr (KS > 1) {
        v4f* const xch =
            reinterpret_cast<v4f*>(lds) + (size_t)(wn * WM + wm) * (KS - 1) * MB * NB * 64 + lane;
        // column n, block m: the partials of the groups that do not own it
#pragma unroll
        for (int n = 0; n < NB; ++n)
            if (n % KS != ks) {
                const int k = ks < n % KS ? ks : ks - 1;
#pragma unroll
                for (int m = 0; m < MB; ++m) xch[((n * MB + m) * (KS - 1) + k) * 64] = acc[m][n];
            }
        __syncthreads();
        if (EPI != kUp && ks >= NB) return;
#pragma unroll
        for (int n = 0; n < NB; ++n)
            if (n % KS == ks) {
#pragma unroll
                for (int m = 0; m < MB; ++m) {
                    v4f s = acc[m][n];
#pragma unroll
                    for (int k = 0; k < KS - 1; ++k) s += xch[((n * MB + m) * (KS - 1) + k) * 64];
                    own[m][n / KS] = s;
                }
            }
    } else {
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
            for (int n = 0; n < NB; ++n) own[m][n] = acc[m][n];
    }

    // the scales come off
    if (!HEAD && !exact) {
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int e = wexp[16 * (mb0 + m) + 4 * g + r] - xn;
#pragma unroll
                for (int j = 0; j < NC; ++j) own[m][j][r] = ldexpf(own[m][j][r], e);
            }
    }
    // the same channels to a split map
    auto store_split = [&](void* base, int q, uint32_t px, const v4f& v) {
        float s[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) s[r] = v[r] * pow2(xn);
        h4 hi, lo;
        split_to(s, hi, lo);
        char* p = static_cast<char*>(base) + ((size_t)(2 * q + (g >> 1)) * HW + px) * 16 + 8 * (g & 1);
        *reinterpret_cast<h4*>(p) = hi;
        *reinterpret_cast<h4*>(p + 8 * HW * 16) = lo;
    };

    if constexpr (HEAD) {
        // The rest of a head on the matrix cores, in the registers of the wave
        // that has its sums:
        //   a = relu(s + b0);  t = relu(W2 a + b2);  out = W4 t + b4.
        // A 1x1 layer's reduction step of 32 channels takes M-blocks 2q and
        // 2q + 1: lane (g, col) holds their channels 16 m + 4 g + r, which is
        // its B operand, the weights being packed in that channel order.  Each
        // pixel's channels are scaled to their largest and split (head_limit).  (The
        // waves sharing the layers through LDS, six barriers a workgroup, took
        // 99 us for the three heads at 256 x 256 against 61, 56 among a forward's
        // launches; two waves a SIMD
        // matter more than what a third shape would save: 85 us where the
        // registers allowed one.)
        const int* const pe = reinterpret_cast<const int*>(lds + S::kParamAt) + wm * head_words(EPI);
        const float* const pb = reinterpret_cast<const float*>(pe);
        auto e_at = [&](int at) { return *reinterpret_cast<const v4i*>(pe + at + 4 * g); };
        auto b_of = [&](int at) { return *reinterpret_cast<const v4f*>(pb + at + 4 * g); };
        const float* const w2 = c.w2[hd];
        const float* const w4 = c.w4[hd];
        const int nout = c.nout[hd], nob = (nout + 15) / 16;
        const uint32_t head4 = split1x1_head_words(nout);
        const __amdgpu_buffer_rsrc_t r4 = rsrc_of(w4 + head4, (uint32_t)nob * 2 * 2048u);
        const uint32_t limit2 = head_limit(reinterpret_cast<const uint32_t*>(w2)[64]);
        const uint32_t limit4 = head_limit(reinterpret_cast<const uint32_t*>(w4)[16 * nob]);
        auto exact16 = [&](const float* w32, int ob, const v4f (&v)[4]) {
            v4f o = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    o = __builtin_amdgcn_mfma_f32_16x16x4f32(
                        w32[((size_t)ob * 16 + 4 * m + r) * 64 + lane], v[m][r], o, 0, 0, 0);
            return o;
        };
        // a pixel's largest magnitude over its 64 channels
        auto px_max = [&](const v4f (&v)[4]) {
            uint32_t m = 0;
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int r = 0; r < 4; ++r) m = umax(m, absbits(v[k][r]));
            m = umax(m, (uint32_t)__shfl_xor((int)m, 16));
            return umax(m, (uint32_t)__shfl_xor((int)m, 32));
        };
        auto operands = [&](const v4f (&v)[4], float sc, h8 (&b)[2][2]) {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                float s[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) s[i] = v[2 * q + (i >> 2)][i & 3] * sc;
                split_to(s, b[q][0], b[q][1]);
            }
        };
        // t of the wave's rows as operands (or, from limit4 on, as fp32 values), its
        // exponents, and the rows that are operands
        v4u tb[NC][4];
        int ex[NC];
        uint32_t split_rows = 0;
        h8 wa[2][2][2];
        if constexpr (EPI == kHeads) w_load(r4, 0, wa[0]);
        if (KS == 1 || ks < NB) {
#pragma unroll
            for (int j = 0; j < NC; ++j) {
                v4f act[4], t[4];
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    const v4i e = e_at(16 * m);
                    const v4f b = b_of(64 + 16 * m);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float v = own[m][j][r];
                        act[m][r] = relu((exact ? v : ldexpf(v, e[r] - xn)) + b[r]);
                    }
                }
                const uint32_t am = px_max(act);
                if (__all(am < limit2)) {
                    const int n = scale_exp(am);
                    h8 b[2][2];
                    operands(act, pow2(n), b);
#pragma unroll
                    for (int mo = 0; mo < 4; ++mo) t[mo] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int p = 0; p < 3; ++p)
#pragma unroll
                        for (int q = 0; q < 2; ++q)
#pragma unroll
                            for (int mo = 0; mo < 4; ++mo)
                                t[mo] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                                    w2v[mo][q][p == 0 ? 1 : 0], b[q][p == 1 ? 1 : 0], t[mo], 0, 0,
                                    0);
#pragma unroll
                    for (int mo = 0; mo < 4; ++mo) {
                        const v4i e = e_at(128 + 16 * mo);
#pragma unroll
                        for (int r = 0; r < 4; ++r) t[mo][r] = ldexpf(t[mo][r], e[r] - n);
                    }
                } else {
#pragma unroll
                    for (int mo = 0; mo < 4; ++mo) t[mo] = exact16(w2 + kHead64 + 4096, mo, act);
                }
#pragma unroll
                for (int mo = 0; mo < 4; ++mo) {
                    const v4f b = b_of(192 + 16 * mo);
#pragma unroll
                    for (int r = 0; r < 4; ++r) t[mo][r] = relu(t[mo][r] + b[r]);
                }
                const uint32_t tm = px_max(t);
                ex[j] = 0;
                if (__all(tm < limit4)) {
                    const int n = scale_exp(tm);
                    h8 b[2][2];
                    operands(t, pow2(n), b);
                    ex[j] = -n;
                    split_rows |= 1u << j;
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        tb[j][i] = __builtin_bit_cast(v4u, b[i >> 1][i & 1]);
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) tb[j][i] = __builtin_bit_cast(v4u, t[i]);
                }
            }
        }
        auto exact_out = [&](int ob, const v4u (&b)[4]) {
            v4f v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = __builtin_bit_cast(v4f, b[i]);
            return exact16(w4 + head4 + (size_t)nob * 1024, ob, v);
        };
        if constexpr (EPI == kHeads) {
            // (Buffer stores, dropped beyond the map and the head's planes by
            // their offset, not by a branch.)
            float* const out = c.hout[hd];
            uint32_t at[NC];
#pragma unroll
            for (int j = 0; j < NC; ++j) {
                const int y = row_of(j);
                at[j] = x < W && y < H ? 4u * (uint32_t)(4 * g * a.HW + y * W + x) : 0xf0000000u;
            }
            auto store16 = [&](int ob, const v4f (&o)[NC]) {
                const int left = nout - 16 * ob;
                const __amdgpu_buffer_rsrc_t ro = rsrc_of(
                    out + (size_t)16 * ob * HW, (uint32_t)(left < 16 ? left : 16) * a.HW * 4u);
                const v4f b = b_of(256 + OUTS + 16 * ob);
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int j = 0; j < NC; ++j)
                        __builtin_amdgcn_raw_buffer_store_b32(
                            __builtin_bit_cast(uint32_t, o[j][r] + b[r]), ro,
                            (int)(at[j] + (uint32_t)r * 4u * a.HW), 0, 0);
            };
            auto block = [&](int ob, const h8 (&w)[2][2]) {
                v4f o[NC];
#pragma unroll
                for (int j = 0; j < NC; ++j) o[j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int p = 0; p < 3; ++p)
#pragma unroll
                    for (int q = 0; q < 2; ++q)
#pragma unroll
                        for (int j = 0; j < NC; ++j)
                            o[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                                w[q][p == 0 ? 1 : 0],
                                __builtin_bit_cast(h8, tb[j][2 * q + (p == 1 ? 1 : 0)]), o[j], 0, 0,
                                0);
                const v4i e = e_at(256 + 16 * ob);
#pragma unroll
                for (int j = 0; j < NC; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[j][r] = ldexpf(o[j][r], e[r] + ex[j]);
                store16(ob, o);
            };
            if (split_rows == (1u << NC) - 1) {
                for (int ob = 0; ob < nob; ob += 2) {
                    w_load(r4, ob + 1 < nob ? ob + 1 : ob, wa[1]);
                    __builtin_amdgcn_sched_barrier(0);
                    block(ob, wa[0]);
                    if (ob + 1 >= nob) break;
                    w_load(r4, ob + 2 < nob ? ob + 2 : ob, wa[0]);
                    __builtin_amdgcn_sched_barrier(0);
                    block(ob + 1, wa[1]);
                }
            } else {
                for (int ob = 0; ob < nob; ++ob) {
                    v4f o[NC];
                    w_load(r4, ob, wa[0]);
#pragma unroll
                    for (int j = 0; j < NC; ++j) {
                        if (split_rows >> j & 1) {
                            v4f v = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                            for (int p = 0; p < 3; ++p)
#pragma unroll
                                for (int q = 0; q < 2; ++q)
                                    v = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                                        wa[0][q][p == 0 ? 1 : 0],
                                        __builtin_bit_cast(h8, tb[j][2 * q + (p == 1 ? 1 : 0)]), v,
                                        0, 0, 0);
                            const v4i e = e_at(256 + 16 * ob);
#pragma unroll
                            for (int r = 0; r < 4; ++r) o[j][r] = ldexpf(v[r], e[r] + ex[j]);
                        } else {
                            o[j] = exact_out(ob, tb[j]);
                        }
                    }
                    store16(ob, o);
                }
            }
        } else {
            // The up-mask head's last layer, the convex upsample of the normals
            // by its 9 x 64 outputs and their normalise: wave sb takes
            // sub-pixels 16 sb .. + 15 of every pixel of the tile, so a lane
            // has all 9 taps of its 4 sub-pixels in registers and no mask is
            // written.  Its weights, 9 blocks of 16 outputs, stay in registers
            // over the rows; the activations come from the waves that have
            // them through LDS.  256 x 256: 75 us (73 among a forward's
            // launches) against 97 for the head
            // writing 151 MB of mask and 42 for the upsample reading them;
            // about half is the upsample's vector arithmetic.
            static_assert(EPI != kUp || S::kWaves == 4, "a quarter of the sub-pixels a wave");
            h8 w9[9][2][2];
#pragma unroll
            for (int n = 0; n < 9; ++n) w_load(r4, 4 * n + wave, w9[n]);
            int* const exl = reinterpret_cast<int*>(lds + S::TH * 4096);
            int* const rowok = reinterpret_cast<int*>(lds + S::TH * (4096 + 64));
            __syncthreads();  // the halo or the partial sums are read
            if (KS == 1 || ks < NB) {
#pragma unroll
                for (int j = 0; j < NC; ++j) {
                    const int row = wn * NB + j * KS + ks;
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        reinterpret_cast<v4u*>(lds)[(row * 4 + i) * 64 + lane] = tb[j][i];
                    if (g == 0) exl[row * 16 + col] = ex[j];
                    if (lane == 0) rowok[4 * row] = split_rows >> j & 1;
                }
            }
            __syncthreads();
            const double eps = c.up_eps;
            const float eps_s = (float)(1.01 * eps);
            const int sub0 = 16 * wave + 4 * g;  // the lane's first sub-pixel
            const int oy0 = sub0 / 8 - c.pad_t, ox = 8 * x + sub0 % 8 - c.pad_l;
            for (int row = 0; row < S::TH && ty0 + row < H; ++row) {
                v4u b[4];
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    b[i] = reinterpret_cast<const v4u*>(lds)[(row * 4 + i) * 64 + lane];
                v4f m[9];
                if (__builtin_amdgcn_readfirstlane(rowok[4 * row])) {
                    const int xe = exl[row * 16 + col];
#pragma unroll
                    for (int n = 0; n < 9; ++n) m[n] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int p = 0; p < 3; ++p)
#pragma unroll
                        for (int q = 0; q < 2; ++q)
#pragma unroll
                            for (int n = 0; n < 9; ++n)
                                m[n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                                    w9[n][q][p == 0 ? 1 : 0],
                                    __builtin_bit_cast(h8, b[2 * q + (p == 1 ? 1 : 0)]), m[n], 0,
                                    0, 0);
#pragma unroll
                    for (int n = 0; n < 9; ++n) {
                        const v4i e = e_at(256 + kSubs * n + 16 * wave);
#pragma unroll
                        for (int r = 0; r < 4; ++r) m[n][r] = ldexpf(m[n][r], e[r] + xe);
                    }
                } else {
#pragma unroll
                    for (int n = 0; n < 9; ++n) m[n] = exact_out(4 * n + wave, b);
                }
                bvml::Taps<3> tp;
                float q_sum = 0.0f;
#pragma unroll
                for (int n = 0; n < 9; ++n) {
                    m[n] += b_of(256 + OUTS + kSubs * n + 16 * wave);
                    const v4f v = reinterpret_cast<const v4f*>(
                        lds + S::kPredAt)[(row + n / 3) * (kTW + 2) + col + n % 3];
#pragma unroll
                    for (int k = 0; k < 3; ++k) tp.v[k][n] = v[k];
                    tp.nrm[n] = v[3];
                    q_sum += v[3];
                }
                tp.flush = bvml::kFlushAbs * q_sum;
                float o[3][4];
                unsigned redo = 0;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float mr[9], res[3];
#pragma unroll
                    for (int n = 0; n < 9; ++n) mr[n] = m[n][r];
                    const bool ok = bvml::fast_subpixel<3>(mr, tp, bvml::kNormalize, eps_s, res);
#pragma unroll
                    for (int k = 0; k < 3; ++k) o[k][r] = res[k];
                    redo |= (ok ? 0u : 1u) << r;
                }
                while (redo) {
                    const int r = __builtin_ctz(redo);
                    redo &= redo - 1;
                    float mr[9], res[3];
#pragma unroll
                    for (int n = 0; n < 9; ++n)
                        mr[n] = r == 0 ? m[n][0] : r == 1 ? m[n][1] : r == 2 ? m[n][2] : m[n][3];
                    bvml::exact_subpixel<3>(mr, tp, true, eps, res);
#pragma unroll
                    for (int rr = 0; rr < 4; ++rr)
#pragma unroll
                        for (int k = 0; k < 3; ++k) o[k][rr] = r == rr ? res[k] : o[k][rr];
                }
                const int oy = 8 * (ty0 + row) + oy0;
                if (x >= W || oy < 0 || oy >= c.out_h) continue;
                float* dst = c.up + (size_t)oy * c.out_w;
                const size_t plane = (size_t)c.out_h * c.out_w;
                if (c.up_vec4) {
                    // (all four columns are inside, or none)
                    if (ox >= 0 && ox < c.out_w)
#pragma unroll
                        for (int k = 0; k < 3; ++k)
                            __builtin_nontemporal_store(
                                v4f{o[k][0], o[k][1], o[k][2], o[k][3]},
                                reinterpret_cast<v4f*>(dst + k * plane + ox));
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (ox + r >= 0 && ox + r < c.out_w)
#pragma unroll
                            for (int k = 0; k < 3; ++k) dst[k * plane + ox + r] = o[k][r];
                }
            }
        }
    } else if constexpr (EPI == kPlain) {
        if (x >= W) return;
#pragma unroll
        for (int j = 0; j < NC; ++j) {
            const int y = row_of(j);
            if (y >= H) continue;
#pragma unroll
            for (int m = 0; m < MB; ++m)
                *reinterpret_cast<v4f*>(c.out + c4_at(mb0 + m, (uint32_t)(y * W + x))) = own[m][j];
        }
    } else if constexpr (EPI == kGates) {
        // M-blocks alternate z, r: block 2i holds z channels 16 i.., 2i + 1
        // the r channels 16 i..; every load goes out before the first store
        // (the compiler cannot know that they do not overlap)
        constexpr int MP = MB / 2;
        static_assert(EPI != kGates || MB % 2 == 0, "z and r blocks in pairs");
        if constexpr (!EARLY) epilogue_loads();
        if (x >= W) return;
        const int q0 = mb0 / 2;
#pragma unroll
        for (int j = 0; j < NC; ++j) {
            const int y = row_of(j);
            if (y >= H) continue;
            const uint32_t px = (uint32_t)(y * W + x);
#pragma unroll
            for (int p = 0; p < MP; ++p) {
                v4f zz, rh;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    zz[r] = sigmoid(own[2 * p][j][r] + ep[0][j][p][r] + eb[0][p][r]);
                    rh[r] = sigmoid(own[2 * p + 1][j][r] + ep[1][j][p][r] + eb[1][p][r]) *
                            ep[2][j][p][r];
                }
                *reinterpret_cast<v4f*>(c.z + c4_at(q0 + p, px)) = zz;
                store_split(c.rs, q0 + p, px, rh);
                if (info->rh32) *reinterpret_cast<v4f*>(c.rh32 + c4_at(q0 + p, px)) = rh;
            }
        }
    } else {
        if constexpr (!EARLY) epilogue_loads();
        if (x >= W) return;
#pragma unroll
        for (int j = 0; j < NC; ++j) {
            const int y = row_of(j);
            if (y >= H) continue;
            const uint32_t px = (uint32_t)(y * W + x);
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                v4f hn;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    hn[r] = gru_mix(ep[1][j][m][r], ep[2][j][m][r],
                                    tanhf(own[m][j][r] + ep[0][j][m][r] + eb[0][m][r]));
                *reinterpret_cast<v4f*>(c.out + c4_at(mb0 + m, px)) = hn;
                store_split(c.outs, mb0 + m, px, hn);
            }
        }
    }
}

template <class S>
__global__ __launch_bounds__(S::kThreads, S::kWavesPerSimd) void conv_kernel(KArgs a) {
    __shared__ __align__(16) char lds[S::kLdsBytes];
    conv_group<S>(a, (int)blockIdx.x, (int)gridDim.x, lds);
}

// Two convolutions that do not depend on each other: the first nb blocks do
// b's, the others a's.
template <class A, class B>
__global__ __launch_bounds__(A::kThreads, 2) void pair_kernel(KArgs a, KArgs b, int nb) {
    static_assert(A::kThreads == B::kThreads, "one block size");
    __shared__ __align__(16) char lds[A::kLdsBytes > B::kLdsBytes ? A::kLdsBytes : B::kLdsBytes];
    const int bx = (int)blockIdx.x;
    if (bx < nb)
        conv_group<B>(b, bx, nb, lds);
    else
        conv_group<A>(a, bx - nb, (int)gridDim.x - nb, lds);
}

// The launch's arguments and workgroups.
template <class S>
long long shape_args(const ConvArgs& c, KArgs& a) {
    a = KArgs{};
    a.c = c;
    a.wblocks = c.wcout / 16;
    a.HW = (uint32_t)((size_t)c.H * c.W);
    a.tiles_x = (c.W + kTW - 1) / kTW;
    a.mgroups = c.cout / (16 * S::MB * S::WM);
    return (long long)a.tiles_x * ((c.H + S::TH - 1) / S::TH) * a.mgroups;
}

template <class S>
hipError_t launch(const ConvArgs& c, hipStream_t stream) {
    KArgs a;
    const long long groups = shape_args<S>(c, a);
    if (groups > INT_MAX) return hipErrorInvalidValue;
    hipLaunchKernelGGL((conv_kernel<S>), dim3((unsigned)groups), dim3(S::kThreads), 0, stream, a);
    return hipGetLastError();
}

template <class A, class B>
hipError_t launch_pair(const ConvArgs& ca, const ConvArgs& cb, hipStream_t stream) {
    KArgs a, b;
    const long long na = shape_args<A>(ca, a), nb = shape_args<B>(cb, b);
    if (na + nb > INT_MAX) return hipErrorInvalidValue;
    hipLaunchKernelGGL((pair_kernel<A, B>), dim3((unsigned)(na + nb)), dim3(A::kThreads), 0, stream,
                       a, b, (int)nb);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Packing the weights: a workgroup per 16-channel block.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void pack_kernel(PackArgs a) {
    const int mb = (int)blockIdx.x, nmb = (int)gridDim.x, taps = a.k * a.k, tid = (int)threadIdx.x;
    const bool one = a.k == 1;
    const int cin = a.c1 - a.c0, cols = cin * taps;
    const size_t stride = (size_t)a.cin * taps;  // of a source row
    __shared__ uint32_t rowmax[16];
    __shared__ const float* rowp[16];
    if (tid < 16) {
        rowmax[tid] = 0;
        const int o = 16 * mb + tid;
        int blk = 0, within = o;
        if (a.interleave) {
            blk = (o >> 4) & 1;
            within = 16 * (o >> 5) + (o & 15);
            if (o >= 32 * (a.rows / 16)) { blk = 2; within = o - 2 * a.rows; }
        } else {
            while (blk < 3 && within >= a.rows) { within -= a.rows; ++blk; }
        }
        rowp[tid] = o < a.out ? a.src[blk] + (size_t)within * stride + (size_t)a.c0 * taps : nullptr;
    }
    __syncthreads();
    for (int i = tid; i < 16 * cols; i += 256) {
        const int r = i / cols;
        if (rowp[r]) atomicMax(&rowmax[r], absbits(rowp[r][i - r * cols]));
    }
    __syncthreads();
    // [exponents | the largest] (0 before this launch)
    int* const head = reinterpret_cast<int*>(a.wp);
    if (tid < 16) {
        const uint32_t m = rowmax[tid];
        head[16 * mb + tid] = m < kInfBits ? -scale_exp(m) : 0;
        atomicMax(reinterpret_cast<uint32_t*>(head) + 16 * nmb, m);
    }
    const bool tail = cin > 64;
    const int steps = one ? 2 : split_steps(a.k, tail);
    uint16_t* sw = reinterpret_cast<uint16_t*>(a.wp + split_head_words(nmb)) + (size_t)mb * steps * 1024;
    for (int i = tid; i < steps * 512; i += 256) {
        const int st = i >> 9, l = (i >> 3) & 63, j = i & 7, g = l >> 4;
        const float* row = rowp[l & 15];
        int at = -1;  // the value's place in the row
        if (one) {
            at = 16 * (2 * st + j / 4) + 4 * g + j % 4;
        } else if (st < 2 * taps) {
            at = (32 * (st / taps) + 8 * g + j) * taps + st % taps;
        } else {
            const int t = st - 2 * taps;
            const int ky = a.k == 5 ? 2 * t + (g >> 1) : g;
            const int kx = (a.k == 5 ? 4 * (g & 1) : 0) + j / 2;
            if (ky < a.k && kx < a.k) at = (64 + j % 2) * taps + ky * a.k + kx;
        }
        const uint32_t m = rowmax[l & 15];
        float v[1] = {row && at >= 0 && m < kInfBits ? row[at] * pow2(scale_exp(m)) : 0.0f};
        typedef _Float16 h1 __attribute__((ext_vector_type(1)));
        h1 hi, lo;
        split_to(v, hi, lo);
        sw[st * 1024 + l * 8 + j] = __builtin_bit_cast(uint16_t, hi);
        sw[st * 1024 + 512 + l * 8 + j] = __builtin_bit_cast(uint16_t, lo);
    }
    float* w32 = a.wp + split_head_words(nmb) + (size_t)nmb * steps * 512;
    const int groups = one ? 16 : split_groups(tail);
    w32 += (size_t)mb * groups * taps * 64;
    for (int i = tid; i < groups * taps * 64; i += 256) {
        const int l = i & 63, t = (i >> 6) % taps, cg = (i >> 6) / taps;
        // (a 1x1 layer's step cg = 4 m + r takes inputs 16 m + 4 g + r)
        const int ch = one ? 16 * (cg >> 2) + 4 * (l >> 4) + (cg & 3) : 4 * cg + (l >> 4);
        const float* row = rowp[l & 15];
        w32[i] = row && ch < cin ? row[ch * taps + t] : 0.0f;
    }
}

__global__ void pack_zero_kernel(float* wp, int nmb) { reinterpret_cast<int*>(wp)[16 * nmb] = 0; }

hipError_t pack(const PackArgs& a, hipStream_t stream) {
    const int nmb = (a.out + 15) / 16;
    hipLaunchKernelGGL(pack_zero_kernel, dim3(1), dim3(1), 0, stream, a.wp, nmb);
    hipLaunchKernelGGL(pack_kernel, dim3((unsigned)nmb), dim3(256), 0, stream, a);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// The first steps of a forward, two launches: the maps of the camera, RayReLU
// of the decoder's normals and the maps' largest magnitudes; then the scales
// from those and the split maps.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void camera_kernel(PrologueArgs a, bool vec4) {
    const uint32_t HW = (uint32_t)a.H * (uint32_t)a.W;
    const uint32_t tid = blockIdx.x * 256u + threadIdx.x, nt = gridDim.x * 256u;
    __shared__ uint32_t red[2][4];
    uint32_t mx[2] = {0, 0};
    for (int k = 0; k < 2; ++k) {
        const float* src = k == 0 ? a.hidden : a.feature;
        const size_t n = (size_t)64 * HW;
        if (vec4) {
            // (8 loads in flight: 8.5 us against 12.7 at 256 x 256)
#pragma unroll 8
            for (size_t i = tid; i < n / 4; i += nt) {
                const v4f v = reinterpret_cast<const v4f*>(src)[i];
                mx[k] = umax(umax(mx[k], absbits(v[0])), umax(absbits(v[1]), umax(absbits(v[2]), absbits(v[3]))));
            }
        } else {
            for (size_t i = tid; i < n; i += nt) mx[k] = umax(mx[k], absbits(src[i]));
        }
    }
    for (uint32_t p = tid; p < HW; p += nt) {
        const int y = (int)(p / (uint32_t)a.W), x = (int)(p - (uint32_t)y * a.W);
        const bvml::Ray3f r = bvml::synth_ray(x, y, a.fu, a.cu, a.fv, a.cv);
        a.ray[p] = r.x;
        a.ray[HW + p] = r.y;
        a.ray[(size_t)2 * HW + p] = r.z;
        a.uv[p] = (float)(((x + 0.5) - a.cu) / a.fu);
        a.uv[HW + p] = (float)(((y + 0.5) - a.cv) / a.fv);
        double ox, oy, oz, inv;
        bvml::ray_relu_ref(a.normal[p], a.normal[HW + p], a.normal[(size_t)2 * HW + p], r.x, r.y,
                           r.z, ox, oy, oz, inv);
        a.pred[p] = (float)ox;
        a.pred[HW + p] = (float)oy;
        a.pred[(size_t)2 * HW + p] = (float)oz;
    }
    for (int k = 0; k < 2; ++k) {
        const uint32_t m = wave_max(mx[k]);
        if ((threadIdx.x & 63) == 0) red[k][threadIdx.x >> 6] = m;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        const uint32_t* r = red[threadIdx.x];
        a.info[64 + threadIdx.x * kMaxBlocks + blockIdx.x] =
            umax(umax(r[0], r[1]), umax(r[2], r[3]));
    }
}

// blockIdx.y: 0 hidden, 1 feature (a thread per 8 channels of a pixel), 2 the
// tails (a thread per pixel).  `blocks`: camera_kernel's; uvmax: the largest
// |u|, |v| of the map.
__global__ __launch_bounds__(256) void split_kernel(PrologueArgs a, int blocks, float uvmax) {
    const uint32_t HW = (uint32_t)a.H * (uint32_t)a.W;
    // the largest weight of the layers that read each map (one with an infinity
    // or a NaN takes fp32 products whatever the scale)
    auto largest = [](const float* w, int mb) {
        return reinterpret_cast<const uint32_t*>(w)[16 * mb];
    };
    auto finite = [](uint32_t m) { return m < kInfBits ? m : 0u; };
    const uint32_t wq = largest(a.w_q, a.mb_q);
    const uint32_t wmax[2] = {umax(umax(finite(largest(a.w_zr, a.mb_zr)), finite(wq)),
                                   finite(largest(a.w_h0, a.mb_h0))),
                              finite(largest(a.w_ctx, a.mb_ctx))};
    __shared__ uint32_t red[2][4];
    uint32_t mx[2];
    for (int k = 0; k < 2; ++k) {
        const uint32_t m = wave_max(
            (int)threadIdx.x < blocks ? a.info[64 + k * kMaxBlocks + threadIdx.x] : 0u);
        if ((threadIdx.x & 63) == 0) red[k][threadIdx.x >> 6] = m;
    }
    __syncthreads();
    int n[2], wide[2];
    for (int k = 0; k < 2; ++k) {
        mx[k] = umax(umax(red[k][0], red[k][1]), umax(red[k][2], red[k][3]));
        const uint32_t all = umax(k == 0 ? umax(mx[k], absbits(1.0f)) : mx[k], absbits(uvmax));
        const uint32_t limit = limit_bits(wmax[k], kBudget) - 1;
        n[k] = scale_exp(all < limit ? all : limit);
        wide[k] = all > limit;
    }
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) {
        Info* info = reinterpret_cast<Info*>(a.info);
        for (int k = 0; k < 2; ++k) {
            info->n[k] = n[k];
            info->wide[k] = wide[k];
        }
        info->rh32 = wide[0] || wq >= kInfBits;
    }
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (blockIdx.y == 2) {
        if (i >= HW) return;
        for (int k = 0; k < 2; ++k) {
            uint32_t* t = k == 0 ? a.th : a.tf;
            const int y = (int)(i / (uint32_t)a.W), x = (int)(i - (uint32_t)y * a.W);
            const float s[2] = {(float)(((x + 0.5) - a.cu) / a.fu) * pow2(n[k]),
                                (float)(((y + 0.5) - a.cv) / a.fv) * pow2(n[k])};
            typedef _Float16 h2 __attribute__((ext_vector_type(2)));
            h2 hi, lo;
            split_to(s, hi, lo);
            t[i] = __builtin_bit_cast(uint32_t, hi);
            t[HW + i] = __builtin_bit_cast(uint32_t, lo);
        }
        return;
    }
    const uint32_t grp = i / HW, px = i - grp * HW;
    if (grp >= 8) return;
    const int k = blockIdx.y;
    const float* src = (k == 0 ? a.hidden : a.feature) + (size_t)8 * grp * HW + px;
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = src[(size_t)j * HW];
    if (k == 0) {
        v4f* d = reinterpret_cast<v4f*>(a.hf);
        d[(size_t)(2 * grp) * HW + px] = v4f{v[0], v[1], v[2], v[3]};
        d[(size_t)(2 * grp + 1) * HW + px] = v4f{v[4], v[5], v[6], v[7]};
    }
    const float sc = pow2(n[k]);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] *= sc;
    h8 hi, lo;
    split_to(v, hi, lo);
    h8* d = reinterpret_cast<h8*>(k == 0 ? a.hs : a.fs);
    d[(size_t)grp * HW + px] = hi;
    d[(size_t)(8 + grp) * HW + px] = lo;
}

hipError_t prologue(const PrologueArgs& a, hipStream_t stream) {
    const size_t hw = (size_t)a.H * a.W;
    const size_t want = (hw * 16 + 255) / 256;  // 4 of the 64 channels a thread
    const int blocks = (int)(want < 1 ? 1 : want > kMaxBlocks ? kMaxBlocks : want);
    const bool vec4 = ((reinterpret_cast<uintptr_t>(a.hidden) |
                        reinterpret_cast<uintptr_t>(a.feature)) & 15u) == 0;
    hipLaunchKernelGGL(camera_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, a, vec4);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    auto big = [](double p, double q) { return p > q || p != p ? p : q; };
    const double uvmax =
        big(big(std::fabs((0.5 - a.cu) / a.fu), std::fabs((a.W - 0.5 - a.cu) / a.fu)),
            big(std::fabs((0.5 - a.cv) / a.fv), std::fabs((a.H - 0.5 - a.cv) / a.fv)));
    hipLaunchKernelGGL(split_kernel, dim3((unsigned)((8 * hw + 255) / 256), 3), dim3(256), 0,
                       stream, a, blocks, (float)uvmax);
    return hipGetLastError();
}

// The shapes of a forward's convolutions by grid size, in 16 x 4 tiles: a small
// grid takes small tiles and splits the reduction over a workgroup's waves, so
// that the chip fills; a large one shares each weight over more pixels.  The
// whole forward in us with each set (tiles):
//            13x19(8) 40x60(40) 48x80(60) 60x80(75) 80x100(140) 90x160(230)
//   Tiny       134      152       183       204        292         402
//   Small      151      163       176       198        267         361
//   Medium     194      208        -        223        254         346
//   Large      377      389        -        388        412         438
//            128x160(320) 160x200(520) 200x200(650) 256x256(1024)
//   Medium     472          727          800          1172
//   Large      486          759          805          1044
// Where the lines lie is measured: Medium against Large 801 and 818 us at 650
// tiles, 830 and 823 at 672, 853 and 848 at 704.
// Gates and heads in one launch (they depend on the same hidden state only):
// 19.1 against 12.0 + 11.0 us at 60x80 (Small), 130 against 76 + 64 us at 256x256
// (116 against 70 + 56 among a forward's launches, the clock up).
//                               K  TAIL  MB NB WM WN KS AD EPI
struct Tiny {
    using Context = Shape<5, true, 4, 2, 1, 1, 4, 2, kPlain>;
    using Gates = Shape<5, false, 2, 2, 1, 1, 4, 4, kGates>;
    using Update = Shape<5, false, 2, 2, 1, 1, 4, 4, kUpdate>;
    using Heads = Shape<3, true, 4, 2, 1, 1, 4, 2, kHeads>;
};
struct Small {
    using Context = Shape<5, true, 4, 4, 1, 1, 4, 2, kPlain>;
    using Gates = Shape<5, false, 2, 4, 1, 1, 4, 4, kGates>;
    using Update = Shape<5, false, 2, 4, 1, 1, 4, 4, kUpdate>;
    using Heads = Shape<3, true, 4, 4, 1, 1, 4, 2, kHeads>;
};
// Small's gates and heads are 7 workgroups a tile, and the chip's 256 CUs hold
// 512 of them: past 73 tiles (512 / 7) gates of twice the channels, 5 a tile, avoid
// a second, nearly empty round (197 against 208 us at 60x80, 75 tiles; 187
// against 180 at 50x72, 65).  Its own second round begins past 102 tiles (512 / 5),
// and the line to Medium, at 110, is a measured one: from 103 tiles to there two
// cards ran Medium faster by up to 5%, a third SmallFull by up to 3% (60x112, 105
// tiles: 241 us SmallFull, 230 Medium; 44x160, 110: 243, 241; the third: 229, 228;
// 230, 236).
struct SmallFull : Small {
    using Gates = Shape<5, false, 4, 4, 1, 1, 4, 2, kGates>;
};
struct Medium {
    using Context = Shape<5, true, 4, 4, 1, 2, 2, 2, kPlain>;
    using Gates = Shape<5, false, 2, 4, 1, 2, 2, 4, kGates>;
    using Update = Shape<5, false, 2, 4, 1, 2, 4, 4, kUpdate>;
    using Heads = Shape<3, true, 4, 4, 1, 2, 2, 2, kHeads>;
};
struct Large {
    using Context = Shape<5, true, 2, 4, 2, 2, 1, 2, kPlain>;
    using Gates = Shape<5, false, 4, 4, 2, 2, 1, 2, kGates>;
    using Update = Shape<5, false, 2, 4, 2, 2, 1, 4, kUpdate>;
    using Heads = Medium::Heads;
};

long long tiles_of(const ConvArgs& c) {
    return (long long)((c.W + kTW - 1) / kTW) * ((c.H + 3) / 4);
}

template <class F>
hipError_t by_size(const ConvArgs& c, F f) {
    const long long tiles = tiles_of(c);
    if (tiles <= 48) return f(Tiny{});
    if (tiles <= 73) return f(Small{});
    if (tiles <= 110) return f(SmallFull{});
    if (tiles <= 640) return f(Medium{});
    return f(Large{});
}

// The up-mask head's tiles: one workgroup a CU at a time (its registers), so the
// fewest rows a workgroup that still fit the chip's 256 CUs in one round (one row:
// 4 workgroups a tile); above that the largest tile.  The whole forward against two
// rows throughout: 130 against 133 us at 13x19, 170 against 173 at 36x96 (54
// tiles), 247 against 253 at 80x100, 334 against 340 at 90x160, 447 against 453 at
// 128x160; four rows at 60x80 take 196 against two's 190.
hipError_t up(const ConvArgs& c, hipStream_t stream) {
    const long long tiles = tiles_of(c);
    if (tiles <= 64) return launch<Shape<3, true, 4, 1, 1, 1, 4, 2, kUp>>(c, stream);
    if (tiles <= 128) return launch<Shape<3, true, 4, 2, 1, 1, 4, 2, kUp>>(c, stream);
    if (tiles <= 256) return launch<Shape<3, true, 4, 4, 1, 1, 4, 2, kUp>>(c, stream);
    return launch<Shape<3, true, 4, 4, 1, 2, 2, 2, kUp>>(c, stream);
}

hipError_t conv(Conv op, const ConvArgs& c, hipStream_t stream) {
    if (op == Conv::Up) return up(c, stream);
    return by_size(c, [&](auto set) {
        using Set = decltype(set);
        switch (op) {
            case Conv::Context: return launch<typename Set::Context>(c, stream);
            case Conv::Gates: return launch<typename Set::Gates>(c, stream);
            case Conv::Update: return launch<typename Set::Update>(c, stream);
            default: return launch<typename Set::Heads>(c, stream);
        }
    });
}

hipError_t gates_heads(const ConvArgs& gates, const ConvArgs& heads, hipStream_t stream) {
    return by_size(gates, [&](auto set) {
        using Set = decltype(set);
        return launch_pair<typename Set::Gates, typename Set::Heads>(gates, heads, stream);
    });
}

constexpr Kernels kTable = {pack, prologue, conv, gates_heads};
struct Register {
    Register() { kernels() = &kTable; }
} const g_register;

}  // namespace
