// The native refiner's own kernels (refiner_conv.hip) as its device path
// (refiner.cpp) sees them: the layouts of the maps and weights they share and
// a table of their launchers.  Private to libbvml_dsine_refine.so.
//
// Maps of C channels over HW pixels:
//   c4     fp32, [C / 4][HW][4]: a pixel's 4 consecutive channels in 16 bytes,
//          as an accumulator block's lane holds them
//   split  halfs, [hi, lo][C / 8][HW][8]: a pixel's 8 consecutive channels in
//          16 bytes, as a matrix-core operand's lane takes them; a value v is
//          (hi + lo) 2^-n with n the map's scale exponent (Info); hi is not
//          finite where v 2^n rounds to 2^16 or more, or is not finite itself
//   tail   halfs, [hi, lo][HW][2]: the uv planes at a split map's scale
// A split map takes the bytes of the fp32 map.
#pragma once

#include <cstddef>
#include <cstdint>

#include <hip/hip_runtime.h>

namespace bvml_refine {

// Per-forward values on the device.  index 0: the hidden state's maps (h,
// r*h and the uv tail beside h), 1: the feature map's (and the tail beside it).
struct Info {
    int n[2];     // scale exponents
    int wide[2];  // 1: a split map may hold values that are not finite
    int rh32;     // 1: the gates write r*h as c4 too: the update may need fp32 products
};
constexpr int kMaxBlocks = 256;  // partial maxima of each map
constexpr size_t kInfoWords = 64 + 2 * kMaxBlocks;

// Packed weights, in 32-bit words (pack).  A convolution over 64 channels (and a
// tail of 2), 16-channel M-blocks mb:
//   [16 mblocks] each output channel's scale exponent e: its weights times
//     2^-e are below 2^15; then the bits of the layer's largest magnitude
//     (from 0x7f800000 on: an infinity or a NaN); padded to a multiple of 64
//     words
//   [mb][step][hi, lo][64 lanes][8 halfs] the split weights: lane l holds
//     output channel 16 mb + l % 16 and, in step c k^2 + tap (c = 0, 1),
//     channels 32 c + 8 (l / 16) + j; in the tail's steps, which come last,
//     tap row and column and channel
//       k = 5: (2 step + l / 32, 4 (l / 16 % 2) + j / 2, 64 + j % 2)
//       k = 3: (l / 16,          j / 2,                  64 + j % 2)
//     with zeros where the row or column lies outside the kernel
//   [mb][4-channel group][tap][64 lanes] the same in fp32: lane l holds output
//     channel 16 mb + l % 16, channel 4 group + l / 16
// A 64-input 1x1 layer: the exponents and the largest, [ob][q 0, 1][hi, lo][64][8
// halfs] with lane l holding output 16 ob + l % 16, input
// 16 (2 q + j / 4) + 4 (l / 16) + j % 4 (the accumulators of two M-blocks as
// they stand), then [ob][m 4][r 4][64 lanes] in fp32, lane l holding output
// 16 ob + l % 16, input 16 m + 4 (l / 16) + r.
constexpr int split_steps(int k, bool tail) { return 2 * k * k + (tail ? (k == 5 ? 3 : 1) : 0); }
constexpr uint32_t split_head_words(int mblocks) {
    return (16u * (uint32_t)mblocks + 1 + 63) / 64 * 64;
}
constexpr int split_groups(bool tail) { return tail ? 17 : 16; }
constexpr size_t split_words(int cout, int k, bool tail) {
    const size_t mb = (size_t)cout / 16;
    return split_head_words((int)mb) + mb * split_steps(k, tail) * 512 +
           mb * k * k * split_groups(tail) * 64;
}
constexpr uint32_t split1x1_head_words(int out) { return split_head_words((out + 15) / 16); }
constexpr size_t split1x1_words(int out) {
    return split1x1_head_words(out) + (size_t)2 * ((out + 15) / 16) * 1024;
}

// Packs one layer's weights from OIHW rows on the device: input channels
// [c0, c1) of `cin`, kernel k; `out` rows taken from up to four sources of
// `rows` each, in order or, with interleave, the first two sources in
// alternating blocks of 16 and then the third.
struct PackArgs {
    const float* src[4];
    int rows, interleave, out, cin, c0, c1, k;
    float* wp;
};

// The first steps of a forward: ray and uv maps, pred = RayReLU(normal, ray),
// the scales, hidden as hf (c4) and hs (split), feature as fs (split), the tails.
struct PrologueArgs {
    const float *normal, *hidden, *feature;  // 3, 64 and 64 planes
    double fu, cu, fv, cv;
    int H, W;
    float *ray, *uv, *pred;     // 3, 2 and 3 planes
    float *hf, *hs, *fs;        // 64-channel maps
    uint32_t *th, *tf;          // tails
    // the packed layers that read the features (ctx) and the hidden state, and
    // their 16-channel blocks
    const float *w_ctx, *w_zr, *w_q, *w_h0;
    int mb_ctx, mb_zr, mb_q, mb_h0;
    uint32_t* info;             // kInfoWords: Info, then (from word 64) partial maxima
};

// One convolution.
struct ConvArgs {
    const void* xs;         // split map, 64 channels
    const float* x32;       // the same map in fp32, for the fp32 products: c4 (context: NCHW;
                            // update: written where info says rh32)
    const uint32_t* tail;   // tail, or NULL
    const float* uv;        // the tail's planes in fp32 (exact)
    const uint32_t* info;
    int which;              // the map's index in Info
    const float* wp;        // packed weights, of wcout channels
    int H, W, cout, wcout;  // (cout <= wcout: the first of them)
    const float* s0;        // gates, update: c4 sums to add
    const float *b0, *b1;   // biases: gates z and r; update q
    const float* hf;        // gates, update: the hidden state, c4
    float* z;               // c4: gates write it, update reads it
    void* rs;               // gates: r*h, split
    float* rh32;            // gates: r*h, c4 (where info says rh32)
    float* out;             // context: c4; update: the new hidden state, c4
    void* outs;             // update: the new hidden state, split
    // heads, per head: the two 1x1 layers packed, the three layers' biases,
    // the output planes (NCHW; up: none) and their count
    const float* w2[4];
    const float* w4[4];
    const float* hb0[4];
    const float* hb2[4];
    const float* b4[4];
    float* hout[4];
    int nout[4];
    // up: the normals (3 planes) to upsample by head 3's output; the
    // normalise's eps; the result's rows from pad_t and columns from pad_l, out_h x out_w; whether it takes
    // 16-byte stores
    const float* pred;
    float* up;
    float up_eps;
    int pad_t, pad_l, out_h, out_w;
    bool up_vec4;
};
// Heads: the first three heads; Up: the up-mask head, the convex upsample and
// its normalise.
enum class Conv { Context, Gates, Update, Heads, Up };

struct Kernels {
    hipError_t (*pack)(const PackArgs&, hipStream_t);
    hipError_t (*prologue)(const PrologueArgs&, hipStream_t);
    hipError_t (*conv)(Conv, const ConvArgs&, hipStream_t);
    // Conv::Gates and Conv::Heads of the same hidden state
    hipError_t (*gates_heads)(const ConvArgs& gates, const ConvArgs& heads, hipStream_t);
};
// Set when refiner_conv.hip is linked in (a build of the host code alone has
// none).
const Kernels*& kernels();

}  // namespace bvml_refine
