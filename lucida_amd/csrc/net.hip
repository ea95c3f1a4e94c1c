// Learned denoiser for gfx950: a 4-level encoder-decoder of 3x3 convolutions
// (channels 32/48/64/96, skip connections, ReLU), BF16 weights and activations
// with FP32 accumulation on the matrix cores, trained on the GPU by this file's
// own forward, backward and Adam kernels. There is no counterpart in the
// reference (its only denoiser is the a-trous filter, crates/core/src/denoise.rs);
// the inputs are the reference's Accum channels (gpu_layout.rs:345).
//
// Convolutions are implicit GEMMs on v_mfma_f32_16x16x32_bf16 with the output
// channels as the GEMM's M side: a wave computes 16 output channels x 16
// consecutive pixels of one row per instruction, the K side walks (tap,
// 16-channel block) pairs. Activations are NHWC BF16, staged in LDS by tile, so
// every lane reads its 8 K-values with one 16-byte read; weights are
// pre-swizzled into per-lane fragments so every wave reads them with one
// coalesced 1 KB load per tile. Pooling, the concatenations and their
// gradients happen inside the convolutions. The input-gradient pass is the same
// kernel over transposed, tap-flipped weights; the weight-gradient pass
// transposes pixel tiles through LDS.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "context.hpp"
#include "net.hpp"
#include "side_stream.hpp"

namespace lucida {
namespace {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ inline float b2f(bf16 v) { return (float)v; }
__device__ inline bf16 f2b(float v) { return (bf16)v; }

// ---------------------------------------------------------------------------
// Output channels of an MFMA tile's rows. Tiles go in pairs of 32 channels: row
// 4g + j of the pair's tile q is channel 32 * pair + 8g + 4q + j, so the lane that
// holds rows 4g .. 4g + 3 of both tiles holds eight consecutive channels (one
// 16-byte store). The last tile of an odd count keeps its rows in order.
// ---------------------------------------------------------------------------
__device__ inline int tile_channel(int mt, int tiles, int row) {
    return (mt | 1) < tiles ? 32 * (mt >> 1) + 8 * (row >> 2) + 4 * (mt & 1) + (row & 3) : 16 * mt + row;
}

// ---------------------------------------------------------------------------
// Weight preparation: FP32 master weights W[tap][ci][co] -> BF16 fragments.
// Fragment (chunk c, m-tile mt, lane l, i) holds A[co][k] with co =
// tile_channel(mt, row l%16) and k = the i-th of 8 consecutive input channels of
// K-block kb = 2c + (l/16)/2, half (l/16)%2. transpose = 1 builds the
// input-gradient weights W'[tap][co][ci] = W[8 - tap][ci][co]. One launch makes
// both for every layer (blockIdx.y = 2 * layer + transpose): as 30 launches of
// 2.5 us each they held up the first pass after every change of the weights
// (training step 1.45 -> 1.32 ms).
// ---------------------------------------------------------------------------
struct PrepLayer {
    int cin, cout;
    uint32_t param, frag[2];  // offsets: weights, forward and transposed fragments
};
struct PrepLayers {
    PrepLayer layer[kNetNumLayers];
};

__global__ void k_wprep(PrepLayers layers, const float* __restrict__ params, bf16* __restrict__ fwd,
                        bf16* __restrict__ bwd) {
    const PrepLayer& L = layers.layer[blockIdx.y >> 1];
    const int transpose = blockIdx.y & 1, cin = L.cin, cout = L.cout;
    const float* W = params + L.param;
    bf16* frag = (transpose ? bwd : fwd) + L.frag[transpose];
    const int in_c = transpose ? cout : cin;     // channels the fragment's K walks
    const int out_c = transpose ? cin : cout;    // channels the fragment's M walks
    const int kbs = 9 * in_c / 16;
    const int chunks = (kbs + 1) / 2;
    const int mts = out_c / 16;
    const int total = chunks * mts * 64 * 8;
    for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < total; e += gridDim.x * blockDim.x) {
        const int i = e & 7, l = (e >> 3) & 63, rest = e >> 9;
        const int mt = rest % mts, c = rest / mts;
        const int g = l >> 4, r = l & 15;
        const int kb = 2 * c + (g >> 1);
        float v = 0.0f;
        if (kb < kbs) {
            const int tap = kb / (in_c / 16), cb = kb % (in_c / 16);
            const int k_ch = cb * 16 + 8 * (g & 1) + i;  // input channel of the GEMM
            const int m_ch = tile_channel(mt, mts, r);    // output channel of the GEMM
            v = transpose ? W[((8 - tap) * cin + m_ch) * cout + k_ch] : W[(tap * cin + k_ch) * cout + m_ch];
        }
        frag[e] = f2b(v);
    }
}

// ---------------------------------------------------------------------------
// Convolution (forward, or input gradient with prepared weights).
//
// A block computes 32 pixels x `rows` rows of all output channels. It stages the
// input tile, with its one-pixel halo and all input channels, in LDS (NHWC; the
// 16-byte octets of a pixel and one pad octet, an odd number, so that the 16
// pixels of a fragment read fall into different banks); its waves split the
// rows (`wn`) and the output tiles (`wm`), and a wave keeps NT tiles of 16 pixels x
// MTW tiles of 16 channels in registers. K walks (tap, 16-channel block) pairs as
// the fragments do, so an output's sequence of MFMAs does not depend on the
// split. Weight fragments come from L2, PF chunks ahead of their use.
//
// The input may be the concatenation of a half-resolution tensor (nearest 2x
// upsampling, the first c_low channels) and a full-resolution one; it is then
// read from the two directly and never written out. The epilogue (EPI) does
// what would otherwise be passes of their own over the output:
//   CONV_FWD        bias and ReLU
//   CONV_FWD_POOL   the same, and the 2x2 average pool of the result to out2
//   CONV_BWD        the ReLU mask of the layer below (its output `mask`)
//   CONV_BWD_SPLIT  the gradient of the concatenation: the first c_split
//                   channels summed over 2x2 and masked, the rest to out2
//   CONV_BWD_UNPOOL the gradient through the pool: a quarter of the result
//                   plus the skip branch's gradient `add` at each of the four
//                   pixels, masked
// Each rounds to BF16 where a separate pass would have read BF16, so results are
// the same bit for bit.
// What bounds it: staging, products and stores share a block's time without
// overlapping inside it, so it lives from the two or three blocks that a CU's
// LDS holds (80 -> 32 channels at 1024 x 1024: 103 us, 57 without staging, 74
// without products). Inference of 1024 x 1024: the fifteen layers with their
// pools and concatenations took 858 us with every wave reading its operands
// from L2 for 32 pixels and the passes apart, and take 470 us so; the passes of
// a training step's backward (masks, pools, concatenations) took 400 us and are
// gone. K loops with a branch per chunk cost 65 us more: every chunk then
// waited for the newest weights.
// ---------------------------------------------------------------------------
enum { CONV_FWD, CONV_FWD_POOL, CONV_BWD, CONV_BWD_SPLIT, CONV_BWD_UNPOOL };
constexpr int CONV_BW = 32;           // a block's pixels per row
constexpr int CONV_LW = CONV_BW + 2;  // with the halo
constexpr int CONV_MAX_KBS = 90;      // K-blocks of 160 input channels
constexpr int CONV_STAGE = 10;        // loads in flight a thread while staging

// An NHWC tensor of c_low + c channels: the first c_low from `low` at half the
// resolution (c_low = 0: none).
struct ConvSource {
    const bf16* low;
    const bf16* src;
    int c_low, c;
};

struct ConvArgs {
    ConvSource in;
    const bf16x8* frag;
    const float* bias;
    bf16* out;
    bf16* out2;
    const bf16* mask;
    const bf16* add;
    int n, h, w;
    int mts;               // output tiles of 16 channels
    int relu, c_split;
    int wm, wn, rows;      // waves along channels and rows; rows per block
    int tiles_x, tiles_y;
};

// Blocks go to the eight XCDs in turn; block b of n works on a tile such that
// each XCD's blocks cover one run of tiles, whose halos then meet in its L2.
__device__ inline int xcd_order(uint32_t b, uint32_t n) {
    const uint32_t per = n / 8, rem = n % 8, x = b % 8;
    return (int)(x * per + min(x, rem) + b / 8);
}

// The value of lane ^ 1 (DPP quad_perm [1, 0, 3, 2]).
__device__ inline float swap_pair(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true));
}

// V consecutive channels from ch of the wave's pixels: acc[t][0 .. V) of its
// NT tiles (row t / 2, columns 16 * (t % 2) + r).
template <int EPI, int NT, int V, class Acc>
__device__ inline void conv_emit(const ConvArgs& a, int img, int y0, int x0, int r, int ch, Acc acc) {
    typedef __bf16 vec __attribute__((ext_vector_type(V)));
    const int cout = a.mts * 16;
    float bias[V];
#pragma unroll
    for (int i = 0; i < V; ++i) bias[i] = a.bias ? a.bias[ch + i] : 0.0f;
#pragma unroll
    for (int rp = 0; rp < NT / 4; ++rp)
#pragma unroll
        for (int xt = 0; xt < 2; ++xt) {
            const int x = x0 + 16 * xt + r, y = y0 + 2 * rp;
            if (x >= a.w) continue;  // whole tiles: widths are multiples of 16
            vec v[2];
#pragma unroll
            for (int k = 0; k < 2; ++k)
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    float s = acc(2 * (2 * rp + k) + xt, i) + bias[i];
                    if ((EPI == CONV_FWD || EPI == CONV_FWD_POOL) && a.relu) s = fmaxf(s, 0.0f);
                    v[k][i] = f2b(s);
                }
            if (EPI == CONV_FWD || EPI == CONV_FWD_POOL || EPI == CONV_BWD) {
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    if (y + k >= a.h) continue;
                    const size_t at = (((size_t)img * a.h + y + k) * a.w + x) * cout + ch;
                    if (EPI == CONV_BWD) {
                        const vec m = *reinterpret_cast<const vec*>(a.mask + at);
#pragma unroll
                        for (int i = 0; i < V; ++i)
                            if (!(b2f(m[i]) > 0.0f)) v[k][i] = f2b(0.0f);
                    }
                    *reinterpret_cast<vec*>(a.out + at) = v[k];
                }
            }
            if (EPI == CONV_FWD_POOL || (EPI == CONV_BWD_SPLIT && ch < a.c_split)) {
                // the 2x2 block of an even lane and its neighbour, summed
                // left to right, top to bottom (pooled sizes are whole)
                float s[V];
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    const float p = b2f(v[0][i]), q = b2f(v[1][i]);
                    s[i] = p + swap_pair(p) + q + swap_pair(q);
                }
                if (!(r & 1) && y < a.h) {
                    const int c2 = EPI == CONV_FWD_POOL ? cout : a.c_split;
                    const size_t at = (((size_t)img * (a.h / 2) + y / 2) * (a.w / 2) + x / 2) * c2 + ch;
                    vec o;
                    if (EPI == CONV_FWD_POOL) {
#pragma unroll
                        for (int i = 0; i < V; ++i) o[i] = f2b(0.25f * s[i]);
                        *reinterpret_cast<vec*>(a.out2 + at) = o;
                    } else {
                        const vec m = *reinterpret_cast<const vec*>(a.mask + at);
#pragma unroll
                        for (int i = 0; i < V; ++i) o[i] = f2b(b2f(m[i]) > 0.0f ? s[i] : 0.0f);
                        *reinterpret_cast<vec*>(a.out + at) = o;
                    }
                }
            }
            if (EPI == CONV_BWD_SPLIT && ch >= a.c_split) {
                const int c2 = cout - a.c_split;
#pragma unroll
                for (int k = 0; k < 2; ++k)
                    if (y + k < a.h)
                        *reinterpret_cast<vec*>(a.out2 + (((size_t)img * a.h + y + k) * a.w + x) * c2 + ch -
                                                a.c_split) = v[k];
            }
            if (EPI == CONV_BWD_UNPOOL) {
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    if (y + k >= a.h) continue;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const size_t at = (((size_t)img * 2 * a.h + 2 * (y + k) + q / 2) * 2 * a.w + 2 * x + q % 2) * cout + ch;
                        const vec d = *reinterpret_cast<const vec*>(a.add + at);
                        const vec m = *reinterpret_cast<const vec*>(a.mask + at);
                        vec o;
#pragma unroll
                        for (int i = 0; i < V; ++i)
                            o[i] = f2b(b2f(m[i]) > 0.0f ? 0.25f * b2f(v[k][i]) + b2f(d[i]) : 0.0f);
                        *reinterpret_cast<vec*>(a.out + at) = o;
                    }
                }
            }
        }
}

// Stages rows by - 1 .. by + rows and columns x0 - 1 .. x0 + CONV_BW of image img
// in `lds`: consecutive threads take consecutive octets of the tile's pixels,
// CONV_STAGE loads in flight a thread.
template <bool CAT>
__device__ inline void conv_stage(const ConvArgs& a, int img, int by, int x0, uint4* lds) {
    const int c = a.in.c, c_low = CAT ? a.in.c_low : 0;
    const int octs = (c_low + c) / 8, S = octs + 1, lrows = a.rows + 2;
    const bf16* lowi = CAT ? a.in.low + (size_t)img * (a.h / 2) * (a.w / 2) * c_low : nullptr;
    const bf16* srci = a.in.src + (size_t)img * a.h * a.w * c;
    const int step_o = blockDim.x % octs, step_p = blockDim.x / octs;
    int o = threadIdx.x % octs, p = threadIdx.x / octs;
    int ry = p / CONV_LW, px = p - ry * CONV_LW;
    while (ry < lrows) {
        uint4 v[CONV_STAGE];
        int at[CONV_STAGE];
#pragma unroll
        for (int k = 0; k < CONV_STAGE; ++k) {
            const int x = x0 - 1 + px, y = by - 1 + ry;
            at[k] = ry < lrows ? (ry * CONV_LW + px) * S + o : -1;
            v[k] = make_uint4(0u, 0u, 0u, 0u);
            if (ry < lrows && x >= 0 && x < a.w && y >= 0 && y < a.h) {
                const bf16* q;
                if (CAT && 8 * o < c_low)
                    q = lowi + (((uint32_t)(y >> 1) * (a.w / 2) + (x >> 1)) * c_low + 8 * o);
                else
                    q = srci + (((uint32_t)y * a.w + x) * c + 8 * o - c_low);
                v[k] = *reinterpret_cast<const uint4*>(q);
            }
            o += step_o;
            px += step_p;
            if (o >= octs) {
                o -= octs;
                ++px;
            }
            while (px >= CONV_LW) {
                px -= CONV_LW;
                ++ry;
            }
        }
#pragma unroll
        for (int k = 0; k < CONV_STAGE; ++k)
            if (at[k] >= 0) lds[at[k]] = v[k];
    }
}

template <int MTW, int NT, int PF, int EPI>
__global__ __launch_bounds__(512) void k_conv(ConvArgs a) {
    static_assert(PF % 2 == 0, "the input fragments alternate between two buffers");
    extern __shared__ uint4 cv_lds[];
    __shared__ int s_off[CONV_MAX_KBS + 1];  // K-block -> octet offset in the tile
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wmi = wv % a.wm, wni = wv / a.wm;
    const int g = lane >> 4, r = lane & 15;
    const int tile = xcd_order(blockIdx.x, gridDim.x);
    const int tx = tile % a.tiles_x, rest = tile / a.tiles_x;
    const int by = (rest % a.tiles_y) * a.rows, img = rest / a.tiles_y;
    const int x0 = tx * CONV_BW;
    const int cin = a.in.c_low + a.in.c;
    const int S = cin / 8 + 1;
    const int cbs = cin / 16, kbs = 9 * cbs, chunks = (kbs + 1) / 2;
    const int mt0 = wmi * MTW;
    // the wave's weight fragments of a chunk (a tile past the last repeats it)
    auto weights = [&](int c, bf16x8(&to)[MTW]) {
#pragma unroll
        for (int m = 0; m < MTW; ++m) to[m] = a.frag[((size_t)c * a.mts + min(mt0 + m, a.mts - 1)) * 64 + lane];
    };
    bf16x8 av[PF][MTW];
#pragma unroll
    for (int i = 0; i < PF; ++i) weights(min(i, chunks - 1), av[i]);
    for (int kb = threadIdx.x; kb <= kbs; kb += blockDim.x) {
        const int tap = kb == kbs ? 8 : kb / cbs, cb = kb == kbs ? 0 : kb % cbs;
        s_off[kb] = (tap / 3 * CONV_LW + tap % 3) * S + 2 * cb;
    }
    if (a.in.c_low)
        conv_stage<true>(a, img, by, x0, cv_lds);
    else
        conv_stage<false>(a, img, by, x0, cv_lds);
    f32x4 acc[NT][MTW];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int m = 0; m < MTW; ++m) acc[t][m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const int wrow = wni * (NT / 2);  // the wave's first row in the tile
    const uint4* bp[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) bp[t] = cv_lds + ((wrow + t / 2) * CONV_LW + 16 * (t % 2) + r) * S + (g & 1);
    __syncthreads();
    // The offsets of the lane's K-blocks are read a group of chunks ahead, the
    // input fragments one chunk ahead.
    int off[PF], off_next[PF];
    auto offsets = [&](int c0, int(&to)[PF]) {
#pragma unroll
        for (int i = 0; i < PF; ++i) to[i] = s_off[min(2 * (c0 + i) + (g >> 1), kbs)];
    };
    uint4 bv[2][NT];
    offsets(0, off);
#pragma unroll
    for (int t = 0; t < NT; ++t) bv[0][t] = bp[t][off[0]];
    auto products = [&](const bf16x8(&w)[MTW], const uint4(&x)[NT]) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int m = 0; m < MTW; ++m)
                acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[m], __builtin_bit_cast(bf16x8, x[t]), acc[t][m],
                                                                    0, 0, 0);
    };
    // Whole groups without a branch: after one the compiler would wait for
    // every load in flight, the next group's weights among them.
    int c0 = 0;
    for (; c0 + PF < chunks; c0 += PF) {
        offsets(c0 + PF, off_next);
#pragma unroll
        for (int i = 0; i < PF; ++i) {
            const int on = i + 1 < PF ? off[i + 1 < PF ? i + 1 : 0] : off_next[0];
#pragma unroll
            for (int t = 0; t < NT; ++t) bv[(i + 1) & 1][t] = bp[t][on];
            products(av[i], bv[i & 1]);
            weights(min(c0 + i + PF, chunks - 1), av[i]);
        }
#pragma unroll
        for (int i = 0; i < PF; ++i) off[i] = off_next[i];
    }
    // The last group, whose weights are loaded. An odd count's missing last
    // K-block has zero weights and takes zeros.
#pragma unroll
    for (int i = 0; i < PF; ++i) {
        const int c = c0 + i;
        if (c < chunks) {
            if (i + 1 < PF && c + 1 < chunks) {
#pragma unroll
                for (int t = 0; t < NT; ++t) bv[(i + 1) & 1][t] = bp[t][off[i + 1 < PF ? i + 1 : 0]];
            }
            if (2 * c + 1 == kbs && g >= 2) {
#pragma unroll
                for (int t = 0; t < NT; ++t) bv[i & 1][t] = make_uint4(0u, 0u, 0u, 0u);
            }
            products(av[i], bv[i & 1]);
        }
    }
    // D: lane holds rows 4g + j of each output tile, pixel column r.
    const int y = by + wrow;
    if (y >= a.h) return;
#pragma unroll
    for (int m = 0; m < MTW; m += 2) {
        const int mt = mt0 + m;
        if (mt >= a.mts) continue;
        if (m + 1 < MTW && mt + 1 < a.mts) {  // a pair (mt0 is even then)
            conv_emit<EPI, NT, 8>(a, img, y, x0, r, 16 * mt + 8 * g,
                                  [&](int t, int i) { return i < 4 ? acc[t][m][i] : acc[t][m + 1 < MTW ? m + 1 : m][i - 4]; });
        } else {
            conv_emit<EPI, NT, 4>(a, img, y, x0, r, tile_channel(mt, a.mts, 4 * g),
                                  [&](int t, int i) { return acc[t][m][i]; });
        }
    }
}

// ---------------------------------------------------------------------------
// Weight gradient: dW[tap][ci][co] = sum_p dpre[p][co] * in[p + off(tap)][ci],
// db[co] = sum_p dpre[p][co]: a product with M = co, N = (tap, ci) and the
// pixels as K. MFMA wants eight K values of one channel in a lane, while the
// tensors are NHWC, so a tile of pixels is transposed on its way into LDS:
// a thread loads eight channels of eight pixels (16 bytes each) and writes
// eight 16-byte octets, one channel's eight pixels each (32 v_perm_b32 for 64
// values). The eight pixels of an octet lie `tw` apart in their row (a tile is
// 8 * tw pixels wide), not side by side: the octet of the neighbouring pixels
// is then the neighbouring 16 bytes, so every tap's shifted operand is one
// aligned 16-byte read, and the input is staged once for all nine taps, with a
// one-pixel halo. Channels lie an odd number of octets apart, so the 16
// channels that a read takes fall into different banks.
//
// A block owns a group of input channels, one 16-channel tile per wave, all
// taps and all output channels (9 * MT accumulators a wave), and one slice of
// the tiles; with few channel tiles `ksplit` waves share one and split its
// K steps, adding up through LDS at the end. Slices store their sums to rows of
// `part` (9 * cin * cout weights, then cout bias sums); k_wgrad_sum adds the
// rows in slice order, so gradients, and the training built on them, are the
// same on every run.
//
// What bounds it: the loads of the two tensors, once per channel group, and
// their latency; the products alone take a few microseconds a layer. Over
// eight 256 x 256 crops the fifteen layers take 0.40 ms; gathering each lane's
// operands from untransposed LDS 16 bits at a time, and staging the input
// once per tap, they took 7.8 ms (the training step 10.05 -> 2.40 ms).
// ---------------------------------------------------------------------------
constexpr int WG_MAX_THREADS = 512;
constexpr size_t WG_LDS = 160 * 1024;  // LDS of a CU
constexpr int WG_CUS = 256;

struct WgradPlan {
    int tw, rows;         // tile: 8 * tw pixels x rows
    int nw, groups;       // channel tiles (waves) per group, groups
    int ksplit, slices;   // waves per channel tile; slices of the tiles
    int tiles_x, tiles_y, tiles;
    int in_stride, dp_stride;  // octets from one channel to the next
    size_t lds;
};

// Eight pixels (16 bytes of channels each) into eight octets (one channel each).
__device__ inline void transpose8(const uint4 (&v)[8], uint4 (&o)[8]) {
    const uint32_t lo = 0x05040100u, hi = 0x07060302u;  // the low, the high halves of two words
#define LUCIDA_PAIR(c, m, sel)                                                              \
    o[c] = make_uint4(__builtin_amdgcn_perm(v[1].m, v[0].m, sel), __builtin_amdgcn_perm(v[3].m, v[2].m, sel), \
                      __builtin_amdgcn_perm(v[5].m, v[4].m, sel), __builtin_amdgcn_perm(v[7].m, v[6].m, sel))
    LUCIDA_PAIR(0, x, lo);
    LUCIDA_PAIR(1, x, hi);
    LUCIDA_PAIR(2, y, lo);
    LUCIDA_PAIR(3, y, hi);
    LUCIDA_PAIR(4, z, lo);
    LUCIDA_PAIR(5, z, hi);
    LUCIDA_PAIR(6, w, lo);
    LUCIDA_PAIR(7, w, hi);
#undef LUCIDA_PAIR
}

// Loads the octets' pixels of image row y, x = x0 + 8 values tw apart, eight
// channels from c0 (a multiple of 8); zeros outside the image.
__device__ inline void load_octets(const ConvSource& t, int c0, int img, int h, int w, int y, int x0, int tw,
                                   uint4 (&v)[8]) {
    const bool row = y >= 0 && y < h;
    const bool low = c0 < t.c_low;
    const int sh = low ? 1 : 0, c = low ? t.c_low : t.c;
    const bf16* base = (low ? t.low + c0 : t.src + (c0 - t.c_low)) +
                       ((size_t)img * (h >> sh) + ((row ? y : 0) >> sh)) * (w >> sh) * c;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int x = x0 + j * tw;
        v[j] = make_uint4(0u, 0u, 0u, 0u);
        if (row && x >= 0 && x < w) v[j] = *reinterpret_cast<const uint4*>(base + (size_t)(x >> sh) * c);
    }
}

template <int MT>
__global__ __launch_bounds__(MT > 4 ? 256 : WG_MAX_THREADS) void k_wgrad(ConvSource in, ConvSource dpre, int h, int w,
                                                          WgradPlan pl, float* __restrict__ part) {
    extern __shared__ uint4 wg_lds[];
    constexpr int cout = MT * 16;
    const int cin = in.c_low + in.c;
    const int tw = pl.tw, hw = tw + 2;
    const int pos_in = (pl.rows + 2) * hw, pos_dp = pl.rows * tw;
    uint4* s_in = wg_lds;                                    // [16 * nw][in_stride]
    uint4* s_dp = wg_lds + (size_t)16 * pl.nw * pl.in_stride;  // [cout][dp_stride]
    const int slice = blockIdx.x / pl.groups, group = blockIdx.x % pl.groups;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int ct = wv % pl.nw, ks = wv / pl.nw;  // channel tile in the group; share of its K steps
    const int g = lane >> 4, r = lane & 15;
    const bool bias_wave = group == 0 && ct == 0;
    f32x4 acc[9][MT], accb[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        accb[m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int t = 0; t < 9; ++t) acc[t][m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    bf16x8 ones;
#pragma unroll
    for (int i = 0; i < 8; ++i) ones[i] = f2b(1.0f);
    const int oct_in = 2 * pl.nw;  // channel octets of the group
    const int items_in = oct_in * pos_in, items = items_in + (cout / 8) * pos_dp;
    for (int tile = slice; tile < pl.tiles; tile += pl.slices) {
        const int tx = tile % pl.tiles_x, rest = tile / pl.tiles_x;
        const int y0 = (rest % pl.tiles_y) * pl.rows, img = rest / pl.tiles_y;
        const int x0 = tx * 8 * tw;
        __syncthreads();  // the previous tile's reads are done
        for (int e = threadIdx.x; e < items; e += blockDim.x) {
            uint4 v[8], o[8];
            uint4* dst;
            int stride;
            if (e < items_in) {
                const int c8 = e % oct_in, p = e / oct_in;
                load_octets(in, group * pl.nw * 16 + 8 * c8, img, h, w, y0 + p / hw - 1, x0 + p % hw - 1, tw, v);
                stride = pl.in_stride;
                dst = s_in + (size_t)(8 * c8) * stride + p;
            } else {
                const int f = e - items_in, c8 = f % (cout / 8), p = f / (cout / 8);
                load_octets(dpre, 8 * c8, img, h, w, y0 + p / tw, x0 + p % tw, tw, v);
                stride = pl.dp_stride;
                dst = s_dp + (size_t)(8 * c8) * stride + p;
            }
            transpose8(v, o);
#pragma unroll
            for (int k = 0; k < 8; ++k) dst[k * stride] = o[k];
        }
        __syncthreads();
        // K steps of 32 pixels: lane group g takes position 4s + g
        for (int s = ks; s < pos_dp / 4; s += pl.ksplit) {
            const int p = 4 * s + g;
            const uint4* a = s_dp + (size_t)r * pl.dp_stride + p;
            const uint4* b = s_in + (size_t)(ct * 16 + r) * pl.in_stride + (p / tw) * hw + p % tw;
            bf16x8 av[MT];
#pragma unroll
            for (int m = 0; m < MT; ++m) av[m] = *reinterpret_cast<const bf16x8*>(a + (size_t)m * 16 * pl.dp_stride);
#pragma unroll
            for (int t = 0; t < 9; ++t) {
                const bf16x8 bv = *reinterpret_cast<const bf16x8*>(b + (t / 3) * hw + t % 3);
#pragma unroll
                for (int m = 0; m < MT; ++m)
                    acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[m], bv, acc[t][m], 0, 0, 0);
            }
            if (bias_wave) {
#pragma unroll
                for (int m = 0; m < MT; ++m)
                    accb[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[m], ones, accb[m], 0, 0, 0);
            }
        }
    }
    // The K shares of a channel tile, added up in order by the first, one
    // output tile at a time (so the staging space is enough).
    f32x4* s_red = reinterpret_cast<f32x4*>(wg_lds) + (size_t)ct * 10 * 64 + lane;
    for (int k = 1; k < pl.ksplit; ++k) {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            __syncthreads();
            if (ks == k) {
                s_red[9 * 64] = accb[m];
#pragma unroll
                for (int t = 0; t < 9; ++t) s_red[t * 64] = acc[t][m];
            }
            __syncthreads();
            if (ks == 0) {
                accb[m] += s_red[9 * 64];
#pragma unroll
                for (int t = 0; t < 9; ++t) acc[t][m] += s_red[t * 64];
            }
        }
    }
    if (ks != 0) return;
    // D[m = co][n = ci]: lane holds co = m*16 + 4g + j, ci = the tile's r.
    float* row = part + (size_t)slice * ((size_t)9 * cin * cout + cout);
    const int ci = (group * pl.nw + ct) * 16 + r;
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m)
            *reinterpret_cast<f32x4*>(row + ((size_t)t * cin + ci) * cout + m * 16 + 4 * g) = acc[t][m];
    if (bias_wave && r == 0) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
            *reinterpret_cast<f32x4*>(row + (size_t)9 * cin * cout + m * 16 + 4 * g) = accb[m];
    }
}

// grad[e] = the sum of part[k][e] over the slices: four threads an element,
// each every fourth slice in ascending order, then the four in order. With one
// thread an element the small layers' few blocks waited for one load after
// another.
__global__ __launch_bounds__(256) void k_wgrad_sum(const float* __restrict__ part, uint32_t row, int slices,
                                                   float* __restrict__ grad) {
    __shared__ float red[256];
    const uint32_t e = blockIdx.x * 64 + (threadIdx.x & 63);
    const int q = threadIdx.x >> 6;
    float acc = 0.0f;
    if (e < row) {
#pragma unroll 8
        for (int k = q; k < slices; k += 4) acc += part[(size_t)k * row + e];
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    if (q == 0 && e < row) grad[e] = ((red[threadIdx.x] + red[threadIdx.x + 64]) + red[threadIdx.x + 128]) + red[threadIdx.x + 192];
}

// ---------------------------------------------------------------------------
// Features and loss.
// ---------------------------------------------------------------------------

// Input features from an Accum film (means): log1p(radiance / albedo) (3),
// albedo (3), normal (3), depth / (1 + depth) (1), log1p of the demodulated
// luminance's standard error (1), log2(samples) / 16 (1), the a-trous
// estimate log1p(filtered / albedo) (3), one zero channel; the a-trous
// estimate again, in FP32, into base_log (3 floats per pixel). With
// `target` non-null also writes the target log1p(ref radiance / albedo) (3
// floats per pixel) from the reference film, demodulated by the INPUT film's
// albedo so inference can remodulate with the same guide.
//
// One launch serves up to FEATURE_FILMS films (blockIdx.z): each one's filtered
// colours and reference film, row width and crop origin, and its place in the
// batch. The filtered colours are read from the filter's own plane, 16 bytes a
// pixel: as an Accum film they were 64 written and a line of 64 read.
constexpr int FEATURE_FILMS = 16;
struct FeatureFilm {
    const GpuAccum *film, *ref;
    const float4* base;  // the demodulated a-trous estimate, per pixel of the film
    int fw, x0, y0, img;
};
struct FeatureFilms {
    FeatureFilm film[FEATURE_FILMS];
};

__global__ void k_features(FeatureFilms films, int cw, int ch, bf16* __restrict__ feat, float* __restrict__ base_log,
                           float* __restrict__ target) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y;
    if (x >= cw || y >= ch) return;
    const FeatureFilm& F = films.film[blockIdx.z];
    const GpuAccum *film = F.film, *ref = F.ref;
    const int fw = F.fw, x0 = F.x0, y0 = F.y0, img = F.img;
    const size_t src = (size_t)(y0 + y) * fw + (x0 + x);
    const float4* a = reinterpret_cast<const float4*>(film + src);
    const float4 a0 = a[0], a1 = a[1], a2 = a[2], a3 = a[3];
    const float ns = fmaxf(a0.w, 1.0f);
    const float inv = 1.0f / ns;
    const float al[3] = {fmaxf(a1.x * inv, 1e-3f), fmaxf(a1.y * inv, 1e-3f), fmaxf(a1.z * inv, 1e-3f)};
    const float rd[3] = {a0.x * inv, a0.y * inv, a0.z * inv};
    const float dep = fmaxf(a1.w * inv, 0.0f);
    float f[16];
    for (int k = 0; k < 3; ++k) f[k] = log1pf(fmaxf(rd[k] / al[k], 0.0f));
    for (int k = 0; k < 3; ++k) f[3 + k] = al[k];
    f[6] = a2.x * inv;
    f[7] = a2.y * inv;
    f[8] = a2.z * inv;
    f[9] = dep / (1.0f + dep);
    // Variance of the per-sample radiance, luminance-weighted, over the mean's
    // standard error, demodulated by the albedo's luminance.
    const float var_l = 0.2126f * fmaxf(a3.x * inv - rd[0] * rd[0], 0.0f) +
                        0.7152f * fmaxf(a3.y * inv - rd[1] * rd[1], 0.0f) +
                        0.0722f * fmaxf(a3.z * inv - rd[2] * rd[2], 0.0f);
    const float al_l = 0.2126f * al[0] + 0.7152f * al[1] + 0.0722f * al[2];
    f[10] = log1pf(sqrtf(var_l * inv) / al_l);
    f[11] = log2f(ns) * (1.0f / 16.0f);
    // The a-trous estimate of the same film, demodulated like channels 0..2:
    // the network predicts a correction to it.
    const float4 b0 = F.base[src];  // remodulated as the filter's film is, then demodulated
    f[12] = log1pf(fmaxf(b0.x * al[0] / al[0], 0.0f));
    f[13] = log1pf(fmaxf(b0.y * al[1] / al[1], 0.0f));
    f[14] = log1pf(fmaxf(b0.z * al[2] / al[2], 0.0f));
    f[15] = 0.0f;
    const size_t dst = ((size_t)img * ch + y) * cw + x;
    // The estimate the output corrects, kept in FP32: in BF16 (8 significant
    // bits) a zero correction could not even reproduce it.
    for (int k = 0; k < 3; ++k) base_log[dst * 3 + k] = f[12 + k];
    bf16x8 lo, hi;
    for (int k = 0; k < 8; ++k) {
        lo[k] = f2b(f[k]);
        hi[k] = f2b(f[8 + k]);
    }
    reinterpret_cast<bf16x8*>(feat + dst * 16)[0] = lo;
    reinterpret_cast<bf16x8*>(feat + dst * 16)[1] = hi;
    if (target) {
        const float4 r0 = reinterpret_cast<const float4*>(ref + src)[0];
        const float rinv = 1.0f / fmaxf(r0.w, 1.0f);
        const float rr[3] = {r0.x * rinv, r0.y * rinv, r0.z * rinv};
        for (int k = 0; k < 3; ++k) target[dst * 3 + k] = log1pf(fmaxf(rr[k] / al[k], 0.0f));
    }
}

// Mean squared error of (output + the FP32 a-trous estimate) against the
// target over the 3 used channels; writes dL/dout (bf16, zero on the
// padding channels) and a per-block partial loss.
__global__ void k_loss(const bf16* __restrict__ out, const float* __restrict__ base_log,
                       const float* __restrict__ target, size_t pixels, bf16* __restrict__ dout,
                       float* __restrict__ loss_partial) {
    __shared__ float red[256];
    float s = 0.0f;
    const float scale = 2.0f / (float)(pixels * 3);
    for (size_t p = (size_t)blockIdx.x * blockDim.x + threadIdx.x; p < pixels; p += (size_t)gridDim.x * blockDim.x) {
        bf16x8 d0, d1;
        for (int k = 0; k < 8; ++k) {
            d0[k] = f2b(0.0f);
            d1[k] = f2b(0.0f);
        }
        for (int k = 0; k < 3; ++k) {
            const float e = (b2f(out[p * 16 + k]) + base_log[p * 3 + k]) - target[p * 3 + k];
            s += e * e;
            d0[k] = f2b(scale * e);
        }
        reinterpret_cast<bf16x8*>(dout + p * 16)[0] = d0;
        reinterpret_cast<bf16x8*>(dout + p * 16)[1] = d1;
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if ((int)threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) loss_partial[blockIdx.x] = red[0];
}

// Remodulated prediction into an Accum-shaped film: radiance =
// expm1(max(out + FP32 a-trous estimate, 0)) * albedo, samples = 1, guides
// copied as means.
__global__ void k_compose(const bf16* __restrict__ out, const float* __restrict__ base_log,
                          const GpuAccum* __restrict__ film, size_t pixels, GpuAccum* __restrict__ dst) {
    const size_t p = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= pixels) return;
    const float4* a = reinterpret_cast<const float4*>(film + p);
    const float4 a1 = a[1], a2 = a[2];
    const float inv = 1.0f / fmaxf(a[0].w, 1.0f);
    const float al[3] = {fmaxf(a1.x * inv, 1e-3f), fmaxf(a1.y * inv, 1e-3f), fmaxf(a1.z * inv, 1e-3f)};
    float rad[3];
    for (int k = 0; k < 3; ++k)
        rad[k] = expm1f(fmaxf(b2f(out[p * 16 + k]) + base_log[p * 3 + k], 0.0f)) * al[k];
    float4* o = reinterpret_cast<float4*>(dst + p);
    o[0] = make_float4(rad[0], rad[1], rad[2], 1.0f);
    o[1] = make_float4(al[0], al[1], al[2], a1.w * inv);
    o[2] = make_float4(a2.x * inv, a2.y * inv, a2.z * inv, 0.0f);
    o[3] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

// Adam (Kingma & Ba) on fp32 parameters; step t >= 1.
__global__ void k_adam(float* __restrict__ p, const float* __restrict__ grad, float* __restrict__ m,
                       float* __restrict__ v, size_t count, float lr, float b1, float b2, float eps, float bc1,
                       float bc2) {
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < count; e += (size_t)gridDim.x * blockDim.x) {
        const float gr = grad[e];
        const float mm = b1 * m[e] + (1.0f - b1) * gr;
        const float vv = b2 * v[e] + (1.0f - b2) * gr * gr;
        m[e] = mm;
        v[e] = vv;
        p[e] -= lr * (mm / bc1) / (sqrtf(vv / bc2) + eps);
    }
}

// The a-trous filter the network corrects: DenoiseParams' defaults
// (crates/core/src/denoise.rs:62-94).
const lucida_denoise_params kAtrousDefaults = {4u, 64.0f, 0.08f, 4.0f, 0.1f};

// Films filtered together for a batch's features, by their pixels: enough to
// fill the device, while the filter's planes stay near 240 MB.
constexpr size_t NET_FILTER_PIXELS = (size_t)1 << 22;

inline unsigned grid1(size_t n, int block = 256) {
    size_t g = (n + block - 1) / block;
    return (unsigned)(g > 65535 * 16 ? 65535 * 16 : (g ? g : 1));
}

}  // namespace

// --- host side --------------------------------------------------------------------

const NetLayer kNetLayers[kNetNumLayers] = {
    {16, 32, 1},  {32, 32, 1},  {32, 48, 1}, {48, 48, 1}, {48, 64, 1}, {64, 64, 1}, {64, 96, 1}, {96, 96, 1},
    {160, 64, 1}, {64, 64, 1},  {112, 48, 1}, {48, 48, 1}, {80, 32, 1}, {32, 32, 1}, {32, 16, 0},
};

// Resolution level of each layer (level k is 2^k smaller per side).
static const int kNetLevel[kNetNumLayers] = {0, 0, 1, 1, 2, 2, 3, 3, 2, 2, 1, 1, 0, 0, 0};

size_t net_param_count() {
    size_t c = 0;
    for (const auto& l : kNetLayers) c += (size_t)9 * l.cin * l.cout + l.cout;
    return c;
}

constexpr size_t CONV_LDS = 160 * 1024 - 512;  // LDS of a CU, less the offset table

// Launches k_conv with the epilogue `epi`, one of those that this split serves.
template <int MTW, int NT, int PF, int... EPI>
static lucida_status launch_conv_t(hipStream_t s, int epi, ConvArgs a, int wm, int wn) {
    a.wm = wm;
    a.wn = wn;
    a.rows = wn * (NT / 2);
    a.tiles_x = (a.w + CONV_BW - 1) / CONV_BW;
    a.tiles_y = (a.h + a.rows - 1) / a.rows;
    const size_t lds = (size_t)(a.rows + 2) * CONV_LW * ((a.in.c_low + a.in.c) / 8 + 1) * 16;
    if (lds > CONV_LDS || wm * wn > 8 || wm * MTW < a.mts || a.in.c_low + a.in.c > CONV_MAX_KBS / 9 * 16)
        return set_error(LUCIDA_INVALID_ARG, "conv: tile larger than a block");
    const dim3 grid(a.n * a.tiles_x * a.tiles_y), block(64 * wm * wn);
    auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, block, lds, s, a); };
    if (!((epi == EPI && (launch(k_conv<MTW, NT, PF, EPI>), true)) || ...))
        return set_error(LUCIDA_INVALID_ARG, "conv: no kernel for this split and epilogue");
    return LUCIDA_OK;
}

// The split by size. From 256 x 256 pixels a wave keeps all output tiles of 64 or
// 128 pixels, as weights are then read least; 128 pixels only where two tiles and
// few input channels leave LDS for it (80 channels: 217 us at 128 pixels, one
// block a CU, 123 us at 64, both at 1024 x 1024); blocks of two waves instead
// of four lose more to the halo than they gain (513 us for all layers against
// 469). Below, and above five output tiles, waves share the tiles in pairs,
// and below 128 x 128 one each, so that the coarse levels still make enough
// waves (96 to 96 channels at 48 x 27: 16 us with 81 waves that keep all
// tiles, 8 us with 168).
static lucida_status launch_conv(hipStream_t s, int epi, const ConvArgs& a) {
    const int mt = a.mts;
    const long px = (long)a.n * a.h * a.w;
    if (mt > 10) return set_error(LUCIDA_INVALID_ARG, "conv: unsupported output channel count");
    if (px < 256L * 256 || mt > 5) {
        if (px < 128L * 128 && mt <= 8)
            return launch_conv_t<1, 4, 8, CONV_FWD, CONV_FWD_POOL, CONV_BWD, CONV_BWD_SPLIT, CONV_BWD_UNPOOL>(s, epi, a,
                                                                                                            mt, 1);
        return launch_conv_t<2, 4, 4, CONV_FWD, CONV_FWD_POOL, CONV_BWD, CONV_BWD_SPLIT, CONV_BWD_UNPOOL>(
            s, epi, a, (mt + 1) / 2, mt <= 4 ? 2 : 1);
    }
    // The concatenations' gradients have 5, 7 and 10 output tiles (layers 12, 10
    // and 8), the last layer's output one.
    switch (mt) {
        case 1: return launch_conv_t<1, 8, 4, CONV_FWD>(s, epi, a, 1, 4);
        case 2:
            if (a.in.c_low + a.in.c > 64) return launch_conv_t<2, 4, 4, CONV_FWD>(s, epi, a, 1, 4);
            return launch_conv_t<2, 8, 2, CONV_FWD, CONV_FWD_POOL, CONV_BWD, CONV_BWD_UNPOOL>(s, epi, a, 1, 4);
        case 3: return launch_conv_t<3, 4, 4, CONV_FWD, CONV_FWD_POOL, CONV_BWD, CONV_BWD_UNPOOL>(s, epi, a, 1, 4);
        case 4: return launch_conv_t<4, 4, 2, CONV_FWD, CONV_FWD_POOL, CONV_BWD, CONV_BWD_UNPOOL>(s, epi, a, 1, 4);
        default: return launch_conv_t<5, 4, 2, CONV_BWD_SPLIT>(s, epi, a, 1, 4);
    }
}

// How a layer's weight gradient is split. Tiles are 64 pixels wide where the
// row allows, else 32 or 16 (rows are multiples of 16). A wave holds 9 * MT
// accumulators of 4 registers, so a block of up to eight waves (256 registers
// each) serves MT up to 4 and one of four waves MT = 6. Few channel tiles
// (16 or 32 channels) share the K steps of larger tiles among more waves.
// Slices: as many blocks as the CUs hold at once (one or two each, by LDS), as
// every slice costs a row of partial sums written and read.
static WgradPlan plan_wgrad(int cin, int cout, int n, int h, int w) {
    WgradPlan p{};
    const int ct = cin / 16, mt = cout / 16;
    const int max_waves = mt > 4 ? 4 : WG_MAX_THREADS / 64;
    p.groups = 1;
    while (ct % p.groups != 0 || ct / p.groups > max_waves) ++p.groups;
    p.nw = ct / p.groups;
    p.ksplit = 1;
    while (p.nw * p.ksplit * 2 <= max_waves) p.ksplit *= 2;
    const int pos = p.ksplit >= 4 ? 64 : 32;  // octets of 8 pixels per tile
    p.tw = w % 64 == 0 ? 8 : (w % 32 == 0 ? 4 : 2);
    p.rows = pos / p.tw;
    p.tiles_x = w / (8 * p.tw);
    p.tiles_y = (h + p.rows - 1) / p.rows;
    p.tiles = n * p.tiles_x * p.tiles_y;
    p.in_stride = ((p.rows + 2) * (p.tw + 2)) | 1;
    p.dp_stride = (p.rows * p.tw) | 1;
    p.lds = (size_t)16 * (16 * p.nw * p.in_stride + cout * p.dp_stride);
    if (p.ksplit > 1) p.lds = std::max(p.lds, (size_t)p.nw * 10 * 1024);
    const int resident = p.lds > WG_LDS / 2 ? 1 : 2;  // blocks a CU
    p.slices = std::max(1, std::min(p.tiles, resident * WG_CUS / p.groups));
    return p;
}

template <int MT>
static lucida_status launch_wgrad_t(hipStream_t s, const ConvSource& in, const bf16* dpre, int h, int w,
                                    const WgradPlan& p, float* part) {
    if (p.lds > WG_LDS) return set_error(LUCIDA_INVALID_ARG, "weight gradient: tile larger than LDS");
    hipLaunchKernelGGL((k_wgrad<MT>), dim3(p.slices * p.groups), dim3(64 * p.nw * p.ksplit), p.lds, s, in,
                       ConvSource{nullptr, dpre, 0, MT * 16}, h, w, p, part);
    return LUCIDA_OK;
}

static lucida_status launch_wgrad(hipStream_t s, const ConvSource& in, const bf16* dpre, int cout, int h, int w,
                                  const WgradPlan& p, float* part) {
    switch (cout / 16) {
        case 1: return launch_wgrad_t<1>(s, in, dpre, h, w, p, part);
        case 2: return launch_wgrad_t<2>(s, in, dpre, h, w, p, part);
        case 3: return launch_wgrad_t<3>(s, in, dpre, h, w, p, part);
        case 4: return launch_wgrad_t<4>(s, in, dpre, h, w, p, part);
        case 6: return launch_wgrad_t<6>(s, in, dpre, h, w, p, part);
        default: return set_error(LUCIDA_INVALID_ARG, "weight gradient: unsupported output channel count");
    }
}

static size_t frag_elems(int in_c, int out_c) {
    const int kbs = 9 * in_c / 16;
    return (size_t)((kbs + 1) / 2) * (out_c / 16) * 64 * 8;
}

}  // namespace lucida

using namespace lucida;

// The network object: fp32 master parameters, Adam moments, bf16 fragments,
// and activation / gradient buffers sized for the largest batch seen.
struct lucida_net {
    lucida_ctx* ctx = nullptr;
    DevBuf params, grads, adam_m, adam_v;  // fp32, layout: per layer W[9][cin][cout] then b[cout]
    DevBuf wg_part;                        // weight-gradient partials: a row of one layer's W and b per slice
    DevBuf frag_fwd, frag_bwd;             // bf16 fragments
    size_t frag_fwd_off[kNetNumLayers], frag_bwd_off[kNetNumLayers], param_off[kNetNumLayers];
    DevBuf acts, dacts, target, loss_partial;
    DevBuf base_log;  // log1p(a-trous estimate / albedo) per pixel of the batch, FP32 (3 floats)
    size_t act_capacity = 0;
    // a gradient ready for its weight gradient; the weight gradients done
    hipEvent_t ev_ready = nullptr, ev_done = nullptr;
    uint32_t step = 0;
    bool frags_valid = false;
    int n = 0, h = 0, w = 0;
};

namespace lucida {

// Activation tensors of one forward pass, as offsets into net->acts.
struct ActPlan {
    size_t x;          // features [n][h][w][16]
    size_t l[15];      // outputs of layers 0..14
    size_t p0, p1, p2; // pooled skip0, skip1, skip2
    size_t total;
};

static ActPlan plan_acts(int n, int h, int w) {
    ActPlan a{};
    size_t off = 0;
    auto take = [&](int hh, int ww, int c) {
        size_t o = off;
        off += (size_t)n * hh * ww * c;
        off = (off + 63) & ~size_t(63);
        return o;
    };
    const int H[4] = {h, h / 2, h / 4, h / 8}, Wd[4] = {w, w / 2, w / 4, w / 8};
    a.x = take(H[0], Wd[0], 16);
    for (int i = 0; i < 15; ++i) a.l[i] = take(H[kNetLevel[i]], Wd[kNetLevel[i]], kNetLayers[i].cout);
    a.p0 = take(H[1], Wd[1], 32);
    a.p1 = take(H[2], Wd[2], 48);
    a.p2 = take(H[3], Wd[3], 64);
    a.total = off;
    return a;
}

// The input of layer li in the activations A: another layer's output, its
// pooled output, or (layers 8, 10 and 12) the layer below upsampled and a skip.
static ConvSource layer_source(const bf16* A, const ActPlan& a, int li) {
    const int cin = kNetLayers[li].cin;
    switch (li) {
        case 0: return ConvSource{nullptr, A + a.x, 0, cin};
        case 2: return ConvSource{nullptr, A + a.p0, 0, cin};
        case 4: return ConvSource{nullptr, A + a.p1, 0, cin};
        case 6: return ConvSource{nullptr, A + a.p2, 0, cin};
        case 8: return ConvSource{A + a.l[7], A + a.l[5], kNetLayers[7].cout, kNetLayers[5].cout};
        case 10: return ConvSource{A + a.l[9], A + a.l[3], kNetLayers[9].cout, kNetLayers[3].cout};
        case 12: return ConvSource{A + a.l[11], A + a.l[1], kNetLayers[11].cout, kNetLayers[1].cout};
        default: return ConvSource{nullptr, A + a.l[li - 1], 0, cin};
    }
}

static lucida_status net_prep_frags(lucida_net* net) {
    hipStream_t s = net->ctx->stream;
    PrepLayers layers;
    for (int i = 0; i < kNetNumLayers; ++i)
        layers.layer[i] = PrepLayer{kNetLayers[i].cin, kNetLayers[i].cout, (uint32_t)net->param_off[i],
                                    {(uint32_t)net->frag_fwd_off[i], (uint32_t)net->frag_bwd_off[i]}};
    hipLaunchKernelGGL(k_wprep, dim3(64, 2 * kNetNumLayers), dim3(256), 0, s, layers, net->params.as<float>(),
                       net->frag_fwd.as<bf16>(), net->frag_bwd.as<bf16>());
    LUCIDA_HIP(hipGetLastError(), LUCIDA_SHADER);
    net->frags_valid = true;
    return LUCIDA_OK;
}

static lucida_status net_ensure_acts(lucida_net* net, int n, int h, int w) {
    if (w % 128 != 0 || h % 8 != 0 || n < 1)
        return set_error(LUCIDA_INVALID_ARG, "denoiser: width must be a multiple of 128 and height of 8");
    ActPlan a = plan_acts(n, h, w);
    if (a.total > net->act_capacity) {
        LUCIDA_HIP(hipStreamSynchronize(net->ctx->stream), LUCIDA_VALIDATION);
        LUCIDA_HIP(net->acts.ensure(a.total * 2), LUCIDA_OOM);
        LUCIDA_HIP(net->dacts.ensure(a.total * 2), LUCIDA_OOM);
        net->act_capacity = a.total;
    }
    LUCIDA_HIP(net->target.ensure((size_t)n * h * w * 3 * 4), LUCIDA_OOM);
    LUCIDA_HIP(net->base_log.ensure((size_t)n * h * w * 3 * 4), LUCIDA_OOM);
    LUCIDA_HIP(net->loss_partial.ensure(4096 * 4), LUCIDA_OOM);
    net->n = n;
    net->h = h;
    net->w = w;
    return LUCIDA_OK;
}

// Forward over the features already in acts[x].
static lucida_status net_forward(lucida_net* net) {
    if (!net->frags_valid) {
        lucida_status st = net_prep_frags(net);
        if (st != LUCIDA_OK) return st;
    }
    hipStream_t s = net->ctx->stream;
    const int n = net->n, H0 = net->h, W0 = net->w;
    const ActPlan a = plan_acts(n, H0, W0);
    bf16* A = net->acts.as<bf16>();
    const float* P = net->params.as<float>();
    const bf16* F = net->frag_fwd.as<bf16>();
    for (int li = 0; li < kNetNumLayers; ++li) {
        const NetLayer& L = kNetLayers[li];
        const int lvl = kNetLevel[li];
        ConvArgs c{};
        c.in = layer_source(A, a, li);
        c.frag = reinterpret_cast<const bf16x8*>(F + net->frag_fwd_off[li]);
        c.bias = P + net->param_off[li] + (size_t)9 * L.cin * L.cout;
        c.relu = L.relu;
        c.out = A + a.l[li];
        c.n = n;
        c.h = H0 >> lvl;
        c.w = W0 >> lvl;
        c.mts = L.cout / 16;
        int epi = CONV_FWD;
        if (li == 1 || li == 3 || li == 5) {  // pooled for the next level
            epi = CONV_FWD_POOL;
            c.out2 = A + (li == 1 ? a.p0 : li == 3 ? a.p1 : a.p2);
        }
        const lucida_status st = launch_conv(s, epi, c);
        if (st != LUCIDA_OK) return st;
    }
    LUCIDA_HIP(hipGetLastError(), LUCIDA_SHADER);
    return LUCIDA_OK;
}

// Backward from dL/dout in dacts[l[14]]; accumulates parameter gradients.
static lucida_status net_backward(lucida_net* net) {
    hipStream_t s = net->ctx->stream;
    const int n = net->n, H0 = net->h, W0 = net->w;
    const ActPlan a = plan_acts(n, H0, W0);
    bf16* A = net->acts.as<bf16>();
    bf16* D = net->dacts.as<bf16>();
    float* G = net->grads.as<float>();
    const bf16* FB = net->frag_bwd.as<bf16>();
    // Every layer's W and b gradients are written whole by its k_wgrad_sum;
    // the partials buffer is sized for the layer with the most.
    WgradPlan wg[kNetNumLayers];
    size_t max_part = 0;
    for (int li = 0; li < kNetNumLayers; ++li) {
        const NetLayer& L = kNetLayers[li];
        wg[li] = plan_wgrad(L.cin, L.cout, n, H0 >> kNetLevel[li], W0 >> kNetLevel[li]);
        max_part = std::max(max_part, (size_t)wg[li].slices * ((size_t)9 * L.cin * L.cout + L.cout));
    }
    if (max_part * 4 > net->wg_part.bytes) {
        LUCIDA_HIP(hipStreamSynchronize(s), LUCIDA_VALIDATION);
        LUCIDA_HIP(net->wg_part.ensure(max_part * 4), LUCIDA_OOM);
    }
    // Every gradient d(layer li) is stored after that layer's ReLU mask. A skip's
    // gradient waits in the d slot of the layer before the skip (l[0], l[2] and
    // l[4], written later) until the pooled branch's is added to it.
    //
    // A layer's weight gradient and its input gradient need only d(layer li):
    // the weight gradients run on a second stream beside the chain of input
    // gradients, since neither fills the device at the coarse levels (training
    // step of eight 256 x 256 crops: 1.32 -> 1.25 ms).
    hipStream_t side = net->ctx->wf[0].s2;
    SideStream beside(s, side, net->ev_ready, net->ev_done);
    for (int li = kNetNumLayers - 1; li >= 0; --li) {
        const NetLayer& L = kNetLayers[li];
        const int lvl = kNetLevel[li];
        LUCIDA_HIP(beside.fork(), LUCIDA_VALIDATION);
        const uint32_t row = (uint32_t)(9 * L.cin * L.cout + L.cout);  // the layer's W then b, as in `grads`
        lucida_status st = launch_wgrad(side, layer_source(A, a, li), D + a.l[li], L.cout, H0 >> lvl, W0 >> lvl, wg[li],
                                        net->wg_part.as<float>());
        if (st != LUCIDA_OK) return st;
        hipLaunchKernelGGL(k_wgrad_sum, dim3((row + 63) / 64), dim3(256), 0, side, net->wg_part.as<float>(), row,
                           wg[li].slices, G + net->param_off[li]);
        if (li == 0) break;
        ConvArgs c{};
        c.in = ConvSource{nullptr, D + a.l[li], 0, L.cout};
        c.frag = reinterpret_cast<const bf16x8*>(FB + net->frag_bwd_off[li]);
        c.n = n;
        c.h = H0 >> lvl;
        c.w = W0 >> lvl;
        c.mts = L.cin / 16;
        c.out = D + a.l[li - 1];
        c.mask = A + a.l[li - 1];
        int epi = CONV_BWD;
        if (li == 8 || li == 10 || li == 12) {  // the upsampled layer below, and a skip
            epi = CONV_BWD_SPLIT;
            c.c_split = kNetLayers[li - 1].cout;
            c.out2 = D + a.l[12 - li];
        } else if (li == 2 || li == 4 || li == 6) {
            epi = CONV_BWD_UNPOOL;
            c.add = D + a.l[li - 2];
        }
        st = launch_conv(s, epi, c);
        if (st != LUCIDA_OK) return st;
    }
    LUCIDA_HIP(beside.join(), LUCIDA_VALIDATION);
    LUCIDA_HIP(hipGetLastError(), LUCIDA_SHADER);
    return LUCIDA_OK;
}

}  // namespace lucida

extern "C" {

lucida_status lucida_net_create(lucida_ctx* ctx, uint32_t seed, lucida_net** out) {
    if (!ctx || !out) return set_error(LUCIDA_INVALID_ARG, "lucida_net_create: null argument");
    auto* net = new lucida_net();
    net->ctx = ctx;
    const size_t np = net_param_count();
    size_t off = 0, ff = 0, fb = 0;
    for (int i = 0; i < kNetNumLayers; ++i) {
        const NetLayer& L = kNetLayers[i];
        net->param_off[i] = off;
        off += (size_t)9 * L.cin * L.cout + L.cout;
        net->frag_fwd_off[i] = ff;
        ff += frag_elems(L.cin, L.cout);
        net->frag_bwd_off[i] = fb;
        fb += frag_elems(L.cout, L.cin);
    }
    // He-normal initialisation from a counter-based stream (Box-Muller over
    // PCG draws); the input's six padding channels and the output's thirteen
    // padding channels start (and, receiving no gradient, stay) at zero. The
    // output layer starts at zero, so an untrained network returns the a-trous
    // estimate it corrects.
    std::vector<float> host(np, 0.0f);
    uint32_t state = seed * 747796405u + 1u;
    auto uni = [&]() {
        state = state * 747796405u + 2891336453u;
        uint32_t word = ((state >> ((state >> 28) + 4u)) ^ state) * 277803737u;
        return ((float)(((word >> 22) ^ word) >> 8) + 0.5f) * (1.0f / 16777216.0f);
    };
    for (int i = 0; i < kNetNumLayers; ++i) {
        const NetLayer& L = kNetLayers[i];
        const int cin_used = i == 0 ? kNetInputsUsed : L.cin;
        const int cout_used = i == kNetNumLayers - 1 ? 3 : L.cout;
        const float stdv = i == kNetNumLayers - 1 ? 0.0f : std::sqrt(2.0f / (9.0f * cin_used));
        float* W = host.data() + net->param_off[i];
        for (int t = 0; t < 9; ++t)
            for (int ci = 0; ci < L.cin; ++ci)
                for (int co = 0; co < L.cout; ++co) {
                    float u1 = uni(), u2 = uni();
                    float z = std::sqrt(-2.0f * std::log(u1)) * std::cos(6.28318530718f * u2);
                    W[(t * L.cin + ci) * L.cout + co] = (ci < cin_used && co < cout_used) ? z * stdv : 0.0f;
                }
    }
    lucida_status st = LUCIDA_OK;
    if (hipEventCreateWithFlags(&net->ev_ready, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&net->ev_done, hipEventDisableTiming) != hipSuccess)
        st = set_error(LUCIDA_VALIDATION, "denoiser event creation failed");
    else if (net->params.ensure(np * 4) != hipSuccess || net->grads.ensure(np * 4) != hipSuccess ||
        net->adam_m.ensure(np * 4) != hipSuccess || net->adam_v.ensure(np * 4) != hipSuccess ||
        net->frag_fwd.ensure(ff * 2) != hipSuccess || net->frag_bwd.ensure(fb * 2) != hipSuccess)
        st = set_error(LUCIDA_OOM, "denoiser parameter allocation failed");
    if (st == LUCIDA_OK &&
        (hipMemcpyAsync(net->params.ptr, host.data(), np * 4, hipMemcpyHostToDevice, ctx->stream) != hipSuccess ||
         hipMemsetAsync(net->adam_m.ptr, 0, np * 4, ctx->stream) != hipSuccess ||
         hipMemsetAsync(net->adam_v.ptr, 0, np * 4, ctx->stream) != hipSuccess ||
         hipMemsetAsync(net->grads.ptr, 0, np * 4, ctx->stream) != hipSuccess ||
         hipStreamSynchronize(ctx->stream) != hipSuccess))
        st = set_error(LUCIDA_VALIDATION, "denoiser parameter upload failed");
    if (st != LUCIDA_OK) {
        lucida_net_destroy(net);
        return st;
    }
    *out = net;
    return LUCIDA_OK;
}

void lucida_net_destroy(lucida_net* net) {
    if (!net) return;
    (void)hipStreamSynchronize(net->ctx->wf[0].s2);
    (void)hipStreamSynchronize(net->ctx->stream);
    if (net->ev_ready) (void)hipEventDestroy(net->ev_ready);
    if (net->ev_done) (void)hipEventDestroy(net->ev_done);
    DevBuf* b[] = {&net->params, &net->grads, &net->adam_m, &net->adam_v, &net->frag_fwd, &net->frag_bwd,
                   &net->acts, &net->dacts, &net->target, &net->loss_partial, &net->base_log,
                   &net->wg_part};
    for (DevBuf* x : b) x->release();
    delete net;
}

size_t lucida_net_param_count(void) { return net_param_count(); }

lucida_status lucida_net_get_params(lucida_net* net, float* out, int which) {
    if (!net || !out || which < 0 || which > 1) return set_error(LUCIDA_INVALID_ARG, "lucida_net_get_params: bad argument");
    const DevBuf& b = which == 0 ? net->params : net->grads;
    LUCIDA_HIP(hipMemcpyAsync(out, b.ptr, net_param_count() * 4, hipMemcpyDeviceToHost, net->ctx->stream),
               LUCIDA_READBACK);
    LUCIDA_HIP(hipStreamSynchronize(net->ctx->stream), LUCIDA_READBACK);
    return LUCIDA_OK;
}

lucida_status lucida_net_set_params(lucida_net* net, const float* in) {
    if (!net || !in) return set_error(LUCIDA_INVALID_ARG, "lucida_net_set_params: null argument");
    LUCIDA_HIP(hipMemcpyAsync(net->params.ptr, in, net_param_count() * 4, hipMemcpyHostToDevice, net->ctx->stream),
               LUCIDA_VALIDATION);
    LUCIDA_HIP(hipStreamSynchronize(net->ctx->stream), LUCIDA_VALIDATION);
    net->frags_valid = false;
    return LUCIDA_OK;
}

// Features of a batch of crops: film k contributes the crop (x0[k], y0[k], w, h).
static lucida_status load_batch(lucida_net* net, const lucida_film* const* inputs, const lucida_film* const* refs,
                                uint32_t count, const uint32_t* x0, const uint32_t* y0, uint32_t w, uint32_t h) {
    if (count > 4096 || w > 16384 || h > 16384 || (uint64_t)count * w * h > (1ull << 26))
        return set_error(LUCIDA_INVALID_ARG, "denoiser: batch larger than 2^26 pixels");
    for (uint32_t k = 0; k < count; ++k) {
        const lucida_film* f = inputs[k];
        if (!f || (refs && !refs[k])) return set_error(LUCIDA_INVALID_ARG, "denoiser: null film");
        const uint64_t cx = x0 ? x0[k] : 0, cy = y0 ? y0[k] : 0;
        if (cx + w > f->width || cy + h > f->height) return set_error(LUCIDA_INVALID_ARG, "crop outside the film");
        if (refs && (refs[k]->width != f->width || refs[k]->height != f->height))
            return set_error(LUCIDA_INVALID_ARG, "reference film size differs");
    }
    lucida_status st = net_ensure_acts(net, (int)count, (int)h, (int)w);
    if (st != LUCIDA_OK) return st;
    // Whole films are filtered (crops then see the filter's real neighbourhood),
    // as many together as make NET_FILTER_PIXELS.
    auto pixels_of = [&](uint32_t k) { return (size_t)inputs[k]->width * inputs[k]->height; };
    auto group_end = [&](uint32_t first, size_t* pixels) {
        uint32_t k = first;
        *pixels = 0;
        while (k < count && (k == first || *pixels + pixels_of(k) <= NET_FILTER_PIXELS)) *pixels += pixels_of(k++);
        return k;
    };
    size_t max_pixels = 0, group = 0;
    for (uint32_t k = 0; k < count;) {
        k = group_end(k, &group);
        max_pixels = std::max(max_pixels, group);
    }
    st = atrous_reserve(net->ctx, max_pixels);
    if (st != LUCIDA_OK) return st;
    const ActPlan a = plan_acts(net->n, net->h, net->w);
    bf16* X = net->acts.as<bf16>() + a.x;
    for (uint32_t first = 0; first < count;) {
        const uint32_t end = group_end(first, &group);
        const float4* filtered = atrous_enqueue(net->ctx, inputs + first, nullptr, end - first, kAtrousDefaults);
        for (uint32_t f0 = first; f0 < end; f0 += FEATURE_FILMS) {
            FeatureFilms ff{};
            const uint32_t n = std::min<uint32_t>(FEATURE_FILMS, end - f0);
            for (uint32_t k = 0; k < n; ++k) {
                ff.film[k] = FeatureFilm{inputs[f0 + k]->accum, refs ? refs[f0 + k]->accum : nullptr, filtered,
                                         (int)inputs[f0 + k]->width, x0 ? (int)x0[f0 + k] : 0,
                                         y0 ? (int)y0[f0 + k] : 0, (int)(f0 + k)};
                filtered += pixels_of(f0 + k);
            }
            hipLaunchKernelGGL(k_features, dim3((w + 127) / 128, h, n), dim3(128), 0, net->ctx->stream, ff, (int)w,
                               (int)h, X, net->base_log.as<float>(), refs ? net->target.as<float>() : nullptr);
        }
        first = end;
    }
    LUCIDA_HIP(hipGetLastError(), LUCIDA_SHADER);
    return LUCIDA_OK;
}

lucida_status lucida_net_forward_backward(lucida_net* net, const lucida_film* const* inputs,
                                          const lucida_film* const* refs, uint32_t count, const uint32_t* x0,
                                          const uint32_t* y0, uint32_t w, uint32_t h, float* loss) {
    if (!net || !inputs || !refs || count == 0) return set_error(LUCIDA_INVALID_ARG, "lucida_net_forward_backward: bad argument");
    clear_error();
    lucida_status st = load_batch(net, inputs, refs, count, x0, y0, w, h);
    if (st != LUCIDA_OK) return st;
    st = net_forward(net);
    if (st != LUCIDA_OK) return st;
    const ActPlan a = plan_acts(net->n, net->h, net->w);
    const size_t pixels = (size_t)net->n * net->h * net->w;
    const unsigned blocks = 1024;
    hipLaunchKernelGGL(k_loss, dim3(blocks), dim3(256), 0, net->ctx->stream, net->acts.as<bf16>() + a.l[14],
                       net->base_log.as<float>(), net->target.as<float>(), pixels, net->dacts.as<bf16>() + a.l[14],
                       net->loss_partial.as<float>());
    st = net_backward(net);
    if (st != LUCIDA_OK) return st;
    if (loss) {
        std::vector<float> part(blocks);
        LUCIDA_HIP(hipMemcpyAsync(part.data(), net->loss_partial.ptr, blocks * 4, hipMemcpyDeviceToHost,
                                  net->ctx->stream),
                   LUCIDA_READBACK);
        LUCIDA_HIP(hipStreamSynchronize(net->ctx->stream), LUCIDA_READBACK);
        double s = 0;
        for (float v : part) s += v;
        *loss = (float)(s / (double)(pixels * 3));
    }
    return LUCIDA_OK;
}

lucida_status lucida_net_adam(lucida_net* net, float lr) {
    if (!net) return set_error(LUCIDA_INVALID_ARG, "lucida_net_adam: null net");
    net->step += 1;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float bc1 = 1.0f - std::pow(b1, (float)net->step), bc2 = 1.0f - std::pow(b2, (float)net->step);
    const size_t np = net_param_count();
    hipLaunchKernelGGL(k_adam, dim3(grid1(np)), dim3(256), 0, net->ctx->stream, net->params.as<float>(),
                       net->grads.as<float>(), net->adam_m.as<float>(), net->adam_v.as<float>(), np, lr, b1, b2, eps,
                       bc1, bc2);
    LUCIDA_HIP(hipGetLastError(), LUCIDA_SHADER);
    return net_prep_frags(net);
}

lucida_status lucida_net_train_step(lucida_net* net, const lucida_film* const* inputs, const lucida_film* const* refs,
                                    uint32_t count, const uint32_t* x0, const uint32_t* y0, uint32_t w, uint32_t h,
                                    float lr, float* loss) {
    lucida_status st = lucida_net_forward_backward(net, inputs, refs, count, x0, y0, w, h, loss);
    if (st != LUCIDA_OK) return st;
    return lucida_net_adam(net, lr);
}

lucida_status lucida_net_denoise(lucida_net* net, const lucida_film* in, lucida_film* out) {
    if (!net || !in || !out) return set_error(LUCIDA_INVALID_ARG, "lucida_net_denoise: null argument");
    if (in == out || in->width != out->width || in->height != out->height)
        return set_error(LUCIDA_INVALID_ARG, "lucida_net_denoise: films must differ and share a size");
    clear_error();
    const lucida_film* ins[1] = {in};
    lucida_status st = load_batch(net, ins, nullptr, 1, nullptr, nullptr, in->width, in->height);
    if (st != LUCIDA_OK) return st;
    st = net_forward(net);
    if (st != LUCIDA_OK) return st;
    const ActPlan a = plan_acts(net->n, net->h, net->w);
    const size_t pixels = (size_t)in->width * in->height;
    hipLaunchKernelGGL(k_compose, dim3(grid1(pixels)), dim3(256), 0, net->ctx->stream, net->acts.as<bf16>() + a.l[14],
                       net->base_log.as<float>(), in->accum, pixels, out->accum);
    LUCIDA_HIP(hipGetLastError(), LUCIDA_SHADER);
    LUCIDA_HIP(hipStreamSynchronize(net->ctx->stream), LUCIDA_VALIDATION);
    return LUCIDA_OK;
}

// Copies one activation tensor of the last forward pass (or its gradient) to
// the host as floats, for parity tests: index 0 = features, 1..15 = layers.
lucida_status lucida_net_read_tensor(lucida_net* net, int index, int gradient, float* out, size_t count) {
    if (!net || !out || index < 0 || index > 15) return set_error(LUCIDA_INVALID_ARG, "lucida_net_read_tensor: bad argument");
    if (net->n == 0) return set_error(LUCIDA_INVALID_ARG, "lucida_net_read_tensor: no forward pass yet");
    const ActPlan a = plan_acts(net->n, net->h, net->w);
    const size_t off = index == 0 ? a.x : a.l[index - 1];
    const int lvl_of[16] = {0, 0, 0, 1, 1, 2, 2, 3, 3, 2, 2, 1, 1, 0, 0, 0};
    const int c = index == 0 ? 16 : kNetLayers[index - 1].cout;
    const int div = 1 << lvl_of[index];
    const size_t want = (size_t)net->n * (net->h / div) * (net->w / div) * c;
    if (count != want) return set_error(LUCIDA_INVALID_ARG, "lucida_net_read_tensor: wrong element count");
    std::vector<uint16_t> tmp(want);
    const DevBuf& b = gradient ? net->dacts : net->acts;
    LUCIDA_HIP(hipMemcpyAsync(tmp.data(), b.as<uint16_t>() + off, want * 2, hipMemcpyDeviceToHost, net->ctx->stream),
               LUCIDA_READBACK);
    LUCIDA_HIP(hipStreamSynchronize(net->ctx->stream), LUCIDA_READBACK);
    for (size_t i = 0; i < want; ++i) {
        uint32_t bits = (uint32_t)tmp[i] << 16;
        std::memcpy(&out[i], &bits, 4);
    }
    return LUCIDA_OK;
}

}  // extern "C"
