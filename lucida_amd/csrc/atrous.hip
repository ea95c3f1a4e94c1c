// Edge-avoiding a-trous denoiser for gfx950.
//
// Reference: shaders/denoise/atrous.wgsl:73-198 with host driver
// crates/gpu/src/denoise.rs:301-408; CPU twin crates/core/src/denoise.rs:134.
// Same algorithm: demodulate by albedo (floored at 1e-3), a 3x3 luminance
// deviation measured once, `iterations` passes of the 5x5 B-spline kernel at
// stride 2^level weighted by normal, depth, luminance and albedo stops, then
// remodulate. Changes for the GPU: the guides are packed once into planes
// (normal + depth, the albedo's luminance) so a tap is 36 bytes instead of a
// 64-byte Accum plus the colour, the colour plane carries its luminance in .w,
// demodulation and deviation are part of the first filter pass and the
// remodulation of the last, each pass filters tiles staged in LDS, and one
// launch per pass serves several films.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "context.hpp"
#include "film_groups.hpp"
#include "shading.hpp"

namespace lucida {
namespace {

using namespace dev;

constexpr int TX = 16, TY = 8;

__device__ inline float lum3(float x, float y, float z) { return x * 0.2126f + y * 0.7152f + z * 0.0722f; }

// The films of one launch: film k (blockIdx.z) has its planes at pixel `base` of
// the context's.
constexpr int DN_JOBS = 16;
struct DnJob {
    const GpuAccum* in;
    GpuAccum* out;
    uint32_t w, h, base, _pad;
};
struct DnJobs {
    DnJob job[DN_JOBS];
};

// Planes over every film's pixels: colour (two, swapped between passes), normal
// and depth, the albedo's luminance, the luminance deviation.
struct DnPlanes {
    float4 *a, *b, *gnd;
    float *alum, *dev;
};

// A pixel of a film: its demodulated colour with luminance, normal and depth,
// and albedo (floored) with luminance.
__device__ inline void dn_pixel(const GpuAccum* __restrict__ in, float4* color, float4* gnd, float4* alb4) {
    const float4* a = reinterpret_cast<const float4*>(in);
    const float4 a0 = a[0], a1 = a[1], a2 = a[2];
    const float inv = 1.0f / fmaxf(a0.w, 1.0f);
    const V3 alb = vmax(V3{a1.x * inv, a1.y * inv, a1.z * inv}, v3s(1.0e-3f));
    const V3 c = V3{a0.x * inv, a0.y * inv, a0.z * inv} / alb;
    *color = make_float4(c.x, c.y, c.z, luminance(c));
    *gnd = make_float4(a2.x * inv, a2.y * inv, a2.z * inv, a1.w * inv);
    *alb4 = make_float4(alb.x, alb.y, alb.z, luminance(alb));
}

// The film's albedo alone, as dn_pixel gives it.
__device__ inline V3 dn_albedo(const GpuAccum* __restrict__ in) {
    const float4* a = reinterpret_cast<const float4*>(in);
    const float4 a1 = a[1];
    const float inv = 1.0f / fmaxf(a[0].w, 1.0f);
    return vmax(V3{a1.x * inv, a1.y * inv, a1.z * inv}, v3s(1.0e-3f));
}

__device__ inline void dn_write(GpuAccum* __restrict__ out, float4 r, V3 al, float4 g) {
    float4* o = reinterpret_cast<float4*>(out);
    o[0] = make_float4(r.x * al.x, r.y * al.y, r.z * al.z, 1.0f);
    o[1] = make_float4(al.x, al.y, al.z, g.w);
    o[2] = make_float4(g.x, g.y, g.z, 0.0f);
    o[3] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

constexpr float LOG2E = 1.4426950408889634f;

// One a-trous pass (atrous.wgsl:129) at a stride of S pixels, S <= 8.
//
// A block filters 64 columns of four rows that lie S apart (one residue of y
// modulo S), staged in LDS with the two rows and 2 * S columns around them
// that its taps reach: rows of one residue see only rows of that residue, so
// wide strides need no taller tile. Pixels outside the image get a zero
// normal, hence weight zero. FIRST (S = 1) reads the film itself, makes the
// guides and the 3x3 luminance deviation (denoise.rs:111) and stores them for
// the later passes; LAST writes the remodulated result (a job without an output
// film leaves the demodulated one in the plane).
//
// The edge stops multiply to one exponential: nd^s * e^-(a+b+c) =
// 2^(s*log2(nd) - (a+b+c)*log2(e)), with the stops' reciprocals taken once per
// pixel and the hardware's exp2 / log2 (a relative error near 1e-6 in a
// weight); every stop must be positive. The hardware's exp2 gives no
// subnormals, so the kernel's factor stays outside it: as part of the exponent
// it made weights vanish that are up to 2^8 times the least. The terms and the
// sums are those of k_dn_pass in its order, so a film's result does not depend
// on which of the two filters it (a pixel outside adds zeros).
//
// What bounds it: vector issue. A tap takes 35 vector instructions, two of them
// at a quarter of the rate; a middle pass at 1024 x 1024 takes 28 us, of which
// the SIMDs issue them for 25, and its LDS reads wait for few bank conflicts
// (0.1M cycles over all CUs). Whole calls at 1024 x 1024: 132 to 142 us, at
// 256 x 256: 37; with every tap read through L1 and the preparation apart, 344 to
// 354 and 54. Fused multiply-adds and the kernel's factor in the exponent would
// take 124 and 35, but give other sums than the untiled passes and lose small
// weights. In that form two or four rows a thread (each tap read from LDS once
// for all of them) left too few waves for the latency: 140 and 145 us against
// 133 on one run, 43 and 61 against 36 at 256 x 256; eight rows a block 136 and
// 37.
constexpr int DN_W = 64, DN_ROWS = 4;
constexpr int DN_THREADS = DN_W * DN_ROWS;
// A grid's y holds 65,535 blocks; 200,000 rows take about 50,000 of 4 rows at
// any stride, and taller films keep the untiled passes (25,000 blocks of 8).
constexpr uint32_t DN_MAX_H = 200000;

template <int S, bool FIRST, bool LAST>
__global__ __launch_bounds__(DN_THREADS) void k_dn_tile(DnJobs jobs, DnPlanes pl, lucida_denoise_params prm) {
    static_assert(!FIRST || S == 1, "the deviation is taken over neighbouring pixels");
    constexpr int PITCH = DN_W + 4 * S, LROWS = DN_ROWS + 4;
    __shared__ float4 s_col[LROWS * PITCH], s_gnd[LROWS * PITCH];
    __shared__ float s_alb[LROWS * PITCH];
    const DnJob& J = jobs.job[blockIdx.z];
    const int w = (int)J.w, h = (int)J.h;
    // the block's residue and first row (counted in strides)
    const int residue = blockIdx.y % S, j0 = (blockIdx.y / S) * DN_ROWS;
    const int x0 = blockIdx.x * DN_W, y0 = residue + j0 * S;
    if (x0 >= w || y0 >= h) return;
    const float4* src = pl.a + J.base;
    float4* gnd = pl.gnd + J.base;
    float* alum = pl.alum + J.base;
    float* dev = pl.dev + J.base;
#pragma unroll 4
    for (int e = threadIdx.x; e < LROWS * PITCH; e += DN_THREADS) {
        const int ly = e / PITCH, lx = e - ly * PITCH;
        const int x = x0 + lx - 2 * S, y = y0 + (ly - 2) * S;
        float4 c = make_float4(0.0f, 0.0f, 0.0f, 0.0f), g = c;
        float al = 0.0f;
        if (x >= 0 && x < w && y >= 0 && y < h) {
            const uint32_t i = (uint32_t)y * J.w + x;
            if (FIRST) {
                float4 a4;
                dn_pixel(J.in + i, &c, &g, &a4);
                al = a4.w;
            } else {
                c = src[i];
                g = gnd[i];
                al = alum[i];
            }
        }
        s_col[e] = c;
        s_gnd[e] = g;
        s_alb[e] = al;
    }
    __syncthreads();
    const int tx = threadIdx.x % DN_W, ty = threadIdx.x / DN_W;
    const int x = x0 + tx, y = y0 + ty * S;
    if (x >= w || y >= h) return;
    const uint32_t i = (uint32_t)y * J.w + x;
    const int at = (ty + 2) * PITCH + tx + 2 * S;
    const float4 cg = s_gnd[at];
    const float cl = s_col[at].w, ca = fmaxf(s_alb[at], 1.0e-3f);
    float d;
    if (FIRST) {
        float sum = 0.0f, sum_sq = 0.0f, n = 0.0f;
        for (int dy = -1; dy <= 1; ++dy)
            for (int dx = -1; dx <= 1; ++dx) {
                const int px = x + dx, py = y + dy;
                if (px < 0 || py < 0 || px >= w || py >= h) continue;
                const float l = s_col[at + dy * PITCH + dx].w;
                sum += l;
                sum_sq += l * l;
                n += 1.0f;
            }
        const float mean = sum / n;
        d = sqrtf(fmaxf(sum_sq / n - mean * mean, 0.0f));
        if (!LAST) {
            gnd[i] = cg;
            alum[i] = s_alb[at];
            dev[i] = d;
        }
    } else {
        d = dev[i];
    }
    const float rd = LOG2E / (prm.sigma_depth * fmaxf(fabsf(cg.w), 1.0e-3f));
    const float rl = LOG2E / (prm.sigma_luminance * fmaxf(d, 1.0e-4f));
    const float ra = LOG2E / (prm.sigma_albedo * ca);
    const float sn = prm.sigma_normal;
    float sx = 0.0f, sy = 0.0f, sz = 0.0f, ws = 0.0f;
#pragma unroll 1
    for (int ky = 0; ky < 5; ++ky) {
        const float kr = ky == 2 ? 3.0f / 8.0f : (ky == 1 || ky == 3 ? 1.0f / 4.0f : 1.0f / 16.0f);
        const float k0 = 1.0f / 16.0f * kr, k1 = 1.0f / 4.0f * kr, k2 = 3.0f / 8.0f * kr;
        const int row = (ty + ky) * PITCH + tx;
#pragma unroll
        for (int kx = 0; kx < 5; ++kx) {
            const float4 qg = s_gnd[row + kx * S];
            const float4 qc = s_col[row + kx * S];
            const float qa = s_alb[row + kx * S];
            const float nd = fmaxf(cg.x * qg.x + cg.y * qg.y + cg.z * qg.z, 0.0f);
            const float ln = sn * __builtin_amdgcn_logf(nd);  // -inf at nd = 0
            const float e = ln - fabsf(cg.w - qg.w) * rd - fabsf(cl - qc.w) * rl - fabsf(ca - qa) * ra;
            const float wt = (kx == 2 ? k2 : (kx == 1 || kx == 3 ? k1 : k0)) * __builtin_amdgcn_exp2f(e);
            sx += qc.x * wt;
            sy += qc.y * wt;
            sz += qc.z * wt;
            ws += wt;
        }
    }
    float4 r = s_col[at];
    if (ws > 0.0f) {
        r.x = sx / ws;
        r.y = sy / ws;
        r.z = sz / ws;
        r.w = lum3(r.x, r.y, r.z);
    }
    if (LAST && J.out)
        dn_write(J.out + i, r, dn_albedo(J.in + i), cg);
    else
        pl.b[J.base + i] = r;
}

// The passes that tiles do not serve (strides of 16 and more, whose halo is
// the larger part of a tile, stops that are not positive, and films of more
// rows than a grid takes) read each tap from the planes.

// The first pass's planes from the film.
__global__ __launch_bounds__(TX* TY) void k_dn_prepare(DnJobs jobs, DnPlanes pl) {
    const DnJob& J = jobs.job[blockIdx.z];
    const uint32_t x = blockIdx.x * TX + threadIdx.x, y = blockIdx.y * TY + threadIdx.y;
    if (x >= J.w || y >= J.h) return;
    const uint32_t i = y * J.w + x;
    float4 al;
    dn_pixel(J.in + i, pl.a + J.base + i, pl.gnd + J.base + i, &al);
    pl.alum[J.base + i] = al.w;
}

// denoise.rs:111 local_deviation: 3x3 luminance standard deviation.
__global__ __launch_bounds__(TX* TY) void k_dn_deviation(DnJobs jobs, DnPlanes pl) {
    const DnJob& J = jobs.job[blockIdx.z];
    const int w = (int)J.w, h = (int)J.h;
    const int x = blockIdx.x * TX + threadIdx.x, y = blockIdx.y * TY + threadIdx.y;
    if (x >= w || y >= h) return;
    const float4* color = pl.a + J.base;
    float sum = 0.0f, sum_sq = 0.0f, n = 0.0f;
    for (int dy = -1; dy <= 1; ++dy)
        for (int dx = -1; dx <= 1; ++dx) {
            const int px = x + dx, py = y + dy;
            if (px < 0 || py < 0 || px >= w || py >= h) continue;
            const float l = color[py * w + px].w;
            sum += l;
            sum_sq += l * l;
            n += 1.0f;
        }
    const float mean = sum / n;
    pl.dev[J.base + y * w + x] = sqrtf(fmaxf(sum_sq / n - mean * mean, 0.0f));
}

__global__ __launch_bounds__(TX* TY) void k_dn_pass(DnJobs jobs, DnPlanes pl, int stride, lucida_denoise_params prm,
                                                    bool last) {
    const DnJob& J = jobs.job[blockIdx.z];
    const int w = (int)J.w, h = (int)J.h;
    const int x = blockIdx.x * TX + threadIdx.x, y = blockIdx.y * TY + threadIdx.y;
    if (x >= w || y >= h) return;
    const float4* src = pl.a + J.base;
    const float4* gnd = pl.gnd + J.base;
    const float* alum = pl.alum + J.base;
    const float K[5] = {1.0f / 16.0f, 1.0f / 4.0f, 3.0f / 8.0f, 1.0f / 4.0f, 1.0f / 16.0f};
    const uint32_t ci = y * w + x;
    const float4 cg = gnd[ci];
    const float4 cc = src[ci];
    const float ca = fmaxf(alum[ci], 1.0e-3f);
    const float lum_scale = prm.sigma_luminance * fmaxf(pl.dev[J.base + ci], 1.0e-4f);
    const float sd = prm.sigma_depth * fmaxf(fabsf(cg.w), 1.0e-3f);
    const float sa = prm.sigma_albedo * ca;
    // one exponential per tap, as in k_dn_tile; nd^0 = 1 also at nd = 0
    const float rd = LOG2E / sd, rl = LOG2E / lum_scale, ra = LOG2E / sa;
    const float sn = prm.sigma_normal;
    float sx = 0.0f, sy = 0.0f, sz = 0.0f, ws = 0.0f;
    for (int ky = 0; ky < 5; ++ky) {
        const int py = y + (ky - 2) * stride;
        if (py < 0 || py >= h) continue;
        for (int kx = 0; kx < 5; ++kx) {
            const int px = x + (kx - 2) * stride;
            if (px < 0 || px >= w) continue;
            const uint32_t qi = py * w + px;
            const float4 qg = gnd[qi];
            const float4 qc = src[qi];
            const float qa = alum[qi];
            const float nd = fmaxf(cg.x * qg.x + cg.y * qg.y + cg.z * qg.z, 0.0f);
            const float ln = sn == 0.0f ? 0.0f : (nd > 0.0f ? sn * __builtin_amdgcn_logf(nd) : -INFINITY);
            const float e = ln - fabsf(cg.w - qg.w) * rd - fabsf(cc.w - qc.w) * rl - fabsf(ca - qa) * ra;
            const float wt = K[kx] * K[ky] * __builtin_amdgcn_exp2f(e);
            sx += qc.x * wt;
            sy += qc.y * wt;
            sz += qc.z * wt;
            ws += wt;
        }
    }
    float4 r = cc;
    if (ws > 0.0f) {
        r.x = sx / ws;
        r.y = sy / ws;
        r.z = sz / ws;
        r.w = lum3(r.x, r.y, r.z);
    }
    if (last && J.out)
        dn_write(J.out + ci, r, dn_albedo(J.in + ci), cg);
    else
        pl.b[J.base + ci] = r;
}

// Zero iterations: remodulate the demodulated colour unchanged.
__global__ __launch_bounds__(TX* TY) void k_dn_modulate(DnJobs jobs) {
    const DnJob& J = jobs.job[blockIdx.z];
    const uint32_t x = blockIdx.x * TX + threadIdx.x, y = blockIdx.y * TY + threadIdx.y;
    if (x >= J.w || y >= J.h) return;
    const uint32_t i = y * J.w + x;
    float4 c, g, al;
    dn_pixel(J.in + i, &c, &g, &al);
    dn_write(J.out + i, c, V3{al.x, al.y, al.z}, g);
}

template <int S>
void launch_tile(uint32_t w, uint32_t h, unsigned jn, hipStream_t s, const DnJobs& jobs, const DnPlanes& pl,
                 const lucida_denoise_params& prm, bool last) {
    const uint32_t rows = DN_ROWS * S;
    const dim3 grid((w + DN_W - 1) / DN_W, S * ((h + rows - 1) / rows), jn);
    if (last)
        hipLaunchKernelGGL((k_dn_tile<S, S == 1, true>), grid, dim3(DN_THREADS), 0, s, jobs, pl, prm);
    else
        hipLaunchKernelGGL((k_dn_tile<S, S == 1, false>), grid, dim3(DN_THREADS), 0, s, jobs, pl, prm);
}

}  // namespace

// Grows the context's a-trous planes to `pixels` (waits for queued work first).
lucida_status atrous_reserve(lucida_ctx* ctx, size_t pixels) {
    const size_t want = pixels * (16 * 3 + 4 * 2);
    if (want > ctx->dn_buf.bytes) {
        LUCIDA_HIP(hipStreamSynchronize(ctx->stream), LUCIDA_VALIDATION);
        LUCIDA_HIP(ctx->dn_buf.ensure(want), LUCIDA_OOM);
    }
    return LUCIDA_OK;
}

// Queues the filter of `count` Accum films on the context's stream, film k into
// `out[k]`; the planes must have been reserved for the films' pixels together.
// With a null `out` (and at least one iteration) the demodulated colours stay in
// a plane of the context, film after film, until its next filter; returned.
const float4* atrous_enqueue(lucida_ctx* ctx, const lucida_film* const* in, GpuAccum* const* out, size_t count,
                    const lucida_denoise_params& params) {
    size_t n = 0;
    for (size_t k = 0; k < count; ++k) n += (size_t)in[k]->width * in[k]->height;
    DnPlanes pl;
    pl.a = ctx->dn_buf.as<float4>();
    pl.b = pl.a + n;
    pl.gnd = pl.b + n;
    pl.alum = reinterpret_cast<float*>(pl.gnd + n);
    pl.dev = pl.alum + n;
    hipStream_t s = ctx->stream;
    size_t base = 0;
    const float4* result = params.iterations % 2 ? pl.b : pl.a;  // the last pass's plane
    unsigned jn;
    for (size_t first = 0; first < count; first += jn) {
        jn = (unsigned)films_together(in + first, count - first, DN_JOBS);
        DnJobs jobs{};
        uint32_t w = 0, h = 0;
        for (unsigned k = 0; k < jn; ++k) {
            const lucida_film* f = in[first + k];
            jobs.job[k] = DnJob{f->accum, out ? out[first + k] : nullptr, f->width, f->height, (uint32_t)base, 0u};
            base += (size_t)f->width * f->height;
            w = std::max(w, f->width);
            h = std::max(h, f->height);
        }
        const dim3 blk(TX, TY), grd((w + TX - 1) / TX, (h + TY - 1) / TY, jn);
        if (params.iterations == 0) {
            hipLaunchKernelGGL(k_dn_modulate, grd, blk, 0, s, jobs);
            continue;
        }
        // stops that are not positive could give a pixel outside the film a weight
        const bool tiles = params.sigma_normal > 0.0f && params.sigma_depth > 0.0f && params.sigma_luminance > 0.0f &&
                           params.sigma_albedo > 0.0f && h <= DN_MAX_H;
        DnPlanes p = pl;
        if (!tiles) {
            hipLaunchKernelGGL(k_dn_prepare, grd, blk, 0, s, jobs, p);
            hipLaunchKernelGGL(k_dn_deviation, grd, blk, 0, s, jobs, p);
        }
        for (uint32_t level = 0; level < params.iterations; ++level) {
            const bool last = level + 1 == params.iterations;
            const uint32_t S = 1u << level;
            if (!tiles || level > 3) hipLaunchKernelGGL(k_dn_pass, grd, blk, 0, s, jobs, p, (int)S, params, last);
            else if (level == 0) launch_tile<1>(w, h, jn, s, jobs, p, params, last);
            else if (level == 1) launch_tile<2>(w, h, jn, s, jobs, p, params, last);
            else if (level == 2) launch_tile<4>(w, h, jn, s, jobs, p, params, last);
            else launch_tile<8>(w, h, jn, s, jobs, p, params, last);
            std::swap(p.a, p.b);
        }
    }
    return result;
}

}  // namespace lucida

using namespace lucida;

extern "C" {

lucida_status lucida_denoise_atrous(lucida_ctx* ctx, const lucida_film* in, const lucida_denoise_params* params,
                                    lucida_film* out) {
    if (!ctx || !in || !params || !out) return set_error(LUCIDA_INVALID_ARG, "lucida_denoise_atrous: null argument");
    if (in == out) return set_error(LUCIDA_INVALID_ARG, "lucida_denoise_atrous: input and output must differ");
    if (in->width != out->width || in->height != out->height)
        return set_error(LUCIDA_INVALID_ARG, "lucida_denoise_atrous: film sizes differ");
    if (params->iterations > 16) return set_error(LUCIDA_INVALID_ARG, "lucida_denoise_atrous: at most 16 iterations");
    clear_error();
    lucida_status st = atrous_reserve(ctx, (size_t)in->width * in->height);
    if (st != LUCIDA_OK) return st;
    atrous_enqueue(ctx, &in, &out->accum, 1, *params);
    LUCIDA_HIP(hipGetLastError(), LUCIDA_SHADER);
    LUCIDA_HIP(hipStreamSynchronize(ctx->stream), LUCIDA_VALIDATION);
    return LUCIDA_OK;
}

}  // extern "C"
