// phiray's a-trous denoiser on gfx950 (src/kernel/denoise.wgsl, driven as
// src/trace/read.rs:85-119 drives it): four passes at tap spacing 1, 2, 4, 8
// over the image buffer, guided by the first hit's albedo, normal and depth and
// by the light itself, the first pass clamping fireflies, the last putting the
// albedo back into the linear sums. One thread per pixel; passes ping-pong
// between the two scratch planes, so a pass never reads what it writes.
// The last pass also writes the display plane and the packed RGBA8 word
// under the camera's view transform, exposure and gamma.
#include "phr_runtime.h"

using namespace phr;

namespace {

// The image buffer as a pass without the guide table reads it, and as the table
// is made: each pixel's guides (sRGB albedo, unit normal, mean depth,
// 1 / count) and the pass's input.
struct Img {
    const uint32_t* __restrict__ px;
    size_t n;
    uint32_t round;
    __device__ float f_at(size_t i) const { return __uint_as_float(px[i]); }
    __device__ V3 v3_at(size_t base, size_t i) const { size_t o = base + 3 * i; return v3(f_at(o), f_at(o + 1), f_at(o + 2)); }
    __device__ float inv_n(size_t i) const {
        uint32_t c = px[31 * n + i];
        return 1.0f / (float)(c > 1u ? c : 1u);
    }
    __device__ static float srgb1(float c) {  // view.wgsl:88-93
        float x = fmin_(fmax_(c, 0.0f), 1.0f);
        float lo = x * 12.92f;
        float hi = 1.055f * dpow(x, 1.0f / 2.4f) - 0.055f;
        return x <= 0.0031308f ? lo : hi;
    }
    __device__ V3 albedo_of(size_t i) const {
        V3 a = v3_at(7 * n, i) * inv_n(i);
        return v3(srgb1(a.x), srgb1(a.y), srgb1(a.z));
    }
    __device__ V3 normal_of(size_t i) const { return normalize(v3_at(10 * n, i) + v3(1e-9f, 1e-9f, 1e-9f)); }
    __device__ float depth_of(size_t i) const { return f_at(13 * n + i) * inv_n(i); }
    __device__ V3 read_in(size_t i) const {
        if (round == 0u) {
            V3 a = v3_at(1 * n, i) * inv_n(i);
            V3 b = vmax(albedo_of(i), 0.05f);
            return v3(a.x / b.x, a.y / b.y, a.z / b.z);
        }
        return v3_at(((round & 1u) == 1u ? 14 : 17) * n, i);
    }
};

__device__ __forceinline__ float luma_of(V3 c) { return dot(c, v3(0.2126f, 0.7152f, 0.0722f)); }

// The last pass's pixel: the albedo put back into the linear sums (unless they
// are kept), the view transform once, under the grid the tracer summed, as the
// tracer composes an unfiltered pixel (denoise.wgsl:124-133). k: 1 / count.
__device__ __forceinline__ void finish_pixel(uint32_t* __restrict__ px, size_t n, size_t i, V3 out, V3 ca, float k, uint32_t keep,
                                             float4 view) {
    const Img im{px, n, 0u};
    const float met = 1.0f - im.f_at(33 * n + i) * k;
    const V3 lin = met > 0.5f * k ? out * vmax(ca, 0.05f) : v3(0, 0, 0);
    if (keep == 0u) {
        const V3 v = lin / k;
        const size_t o = 1 * n + 3 * i;
        px[o] = __float_as_uint(v.x);
        px[o + 1] = __float_as_uint(v.y);
        px[o + 2] = __float_as_uint(v.z);
    }
    const float cov = im.f_at(23 * n + i) * k;
    const V3 grid = im.v3_at(20 * n, i) * k;
    const V3 shown = view_transform(lin / fmax_(met, k), view.x, view.y, view.z, view.w) * (1.0f - cov) + grid;
    px[4 * n + 3 * i] = __float_as_uint(shown.x);
    px[4 * n + 3 * i + 1] = __float_as_uint(shown.y);
    px[4 * n + 3 * i + 2] = __float_as_uint(shown.z);
    px[i] = pack_rgba8(shown, im.f_at(24 * n + i) * k);
}

// The guide table and the first pass's input, once a denoise.
__global__ __launch_bounds__(256) void k_denoise_prep(const uint32_t* __restrict__ px, size_t n, float4* __restrict__ feat,
                                                      float* __restrict__ col0) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const Img im{px, n, 0u};
    const V3 a = im.albedo_of(i), nr = im.normal_of(i), c = im.read_in(i);
    feat[2 * i] = make_float4(a.x, a.y, a.z, im.depth_of(i));
    feat[2 * i + 1] = make_float4(nr.x, nr.y, nr.z, im.inv_n(i));
    col0[3 * i] = c.x;
    col0[3 * i + 1] = c.y;
    col0[3 * i + 2] = c.z;
}

// A pass that derives the guides at every tap: the `denoise` kernel of a
// recorded Pass, and a denoise without scratch.
__global__ __launch_bounds__(256) void k_denoise(uint32_t* __restrict__ px, uint32_t w, uint32_t h, uint32_t step, uint32_t round,
                                                 uint32_t last, uint32_t keep, float s0, float s1, float s2, float s3,
                                                 float4 view) {
    const size_t n = (size_t)w * h;
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float KERNEL[3] = {0.375f, 0.25f, 0.0625f};
    Img im{px, n, round};
    int x = (int)(i % w), y = (int)(i / w);
    V3 centre = im.read_in(i);
    if (round == 0u) {
        float near_top = 0.0f, near_n = 0.0f;
        V3 near_sum = v3(0, 0, 0);
        for (int dy = -1; dy <= 1; ++dy)
            for (int dx = -1; dx <= 1; ++dx) {
                int sx = x + dx, sy = y + dy;
                if ((dx == 0 && dy == 0) || sx < 0 || sy < 0 || sx >= (int)w || sy >= (int)h) continue;
                V3 c = im.read_in((size_t)sy * w + sx);
                near_top = fmax_(near_top, luma_of(c));
                near_sum = near_sum + c;
                near_n = near_n + 1.0f;
            }
        if (near_n > 0.0f && luma_of(centre) > 1.5f * near_top + 0.05f) centre = near_sum / near_n;
    }
    V3 cn = im.normal_of(i), ca = im.albedo_of(i);
    float cd = im.depth_of(i), lc = luma_of(centre);
    V3 sum = v3(0, 0, 0);
    float weight = 0.0f;
    for (int dy = -2; dy <= 2; ++dy)
        for (int dx = -2; dx <= 2; ++dx) {
            int sx = x + dx * (int)step, sy = y + dy * (int)step;
            if (sx < 0 || sy < 0 || sx >= (int)w || sy >= (int)h) continue;
            size_t j = (size_t)sy * w + sx;
            if ((im.depth_of(j) < 0.0f) != (cd < 0.0f)) continue;
            V3 tap = (j == i) ? centre : im.read_in(j);
            float dn = fmax_(0.0f, 1.0f - dot(cn, im.normal_of(j)));
            V3 dav = im.albedo_of(j) - ca;
            float da = sqrtf(dot(dav, dav));
            float dd = fabsf(im.depth_of(j) - cd) / fmax_(fabsf(cd), 1e-3f);
            float dl = fabsf(luma_of(tap) - lc) / (0.08f + lc);
            float stop = dexp(-dn * s0 - da * s1 - dd * s2 - dl * dl * s3);
            float k = KERNEL[dx < 0 ? -dx : dx] * KERNEL[dy < 0 ? -dy : dy];
            sum = sum + tap * k * stop;
            weight = weight + k * stop;
        }
    V3 out = weight > 0.0f ? sum / weight : centre;
    if (last == 0u) {
        size_t o = ((round & 1u) == 1u ? 17 : 14) * n + 3 * i;
        px[o] = __float_as_uint(out.x);
        px[o + 1] = __float_as_uint(out.y);
        px[o + 2] = __float_as_uint(out.z);
        return;
    }
    finish_pixel(px, n, i, out, ca, im.inv_n(i), keep, view);
}

struct Px3 {
    float x, y, z;
};
__device__ __forceinline__ V3 load3(const float* p) {
    const Px3 v = *(const Px3*)p;
    return v3(v.x, v.y, v.z);
}
__device__ __forceinline__ void store3(float* p, V3 v) { *(Px3*)p = Px3{v.x, v.y, v.z}; }

// One pass over the guide table. A lane filters ROWS pixels of one column,
// `step` rows apart, and reads each of the taps they share once: 7 x 5 taps of
// 44 bytes for three pixels, not 75. The arithmetic: the centre's
// divisors are inverted once, the stops' exponent is summed in powers of two
// and taken with the hardware's exp2 and square root (each within an ulp).
// Bound by the arithmetic at three rows (about 40 issue slots a tap, a pass of
// 1080p at 75 us where 198 us were), by the taps' loads at one (192 us). Few
// pixels want more waves instead: us for all four passes at 1 / 2 / 3 / 4 rows:
// 256 x 256 68 / 79 / 97 / 116, 512 x 512 116 / 90 / 110 / 118, 1024 x 512 205 /
// 123 / 138 / 150, 1280 x 720 355 / 202 / 189 / 205, 1920 x 1080 770 / 427 / 378 /
// 387.
constexpr size_t ROWS2_MIN = 163840, ROWS3_MIN = 786432;
constexpr float LOG2E = 1.4426950408889634f;
__device__ __forceinline__ float dotf(V3 a, V3 b) { return __builtin_fmaf(a.x, b.x, __builtin_fmaf(a.y, b.y, a.z * b.z)); }
template <int ROWS, bool FIRST, bool LAST>
__global__ __launch_bounds__(256) void k_atrous(uint32_t* __restrict__ px, uint32_t w, uint32_t h, uint32_t log2_step, uint32_t keep,
                                                float4 strengths, float4 view, const float4* __restrict__ feat,
                                                const float* __restrict__ in, float* __restrict__ out) {
    const int step = 1 << log2_step;
    const int x = (int)(blockIdx.x * 64u + (threadIdx.x & 63u));
    // The rows of a set are y0, y0 + step, ...: a wave's, so scalar.
    const uint32_t set = blockIdx.y * 4u + (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int y0 = (int)(((set >> log2_step) * ROWS << log2_step) + (set & (uint32_t)(step - 1)));
    if (y0 >= (int)h) return;
    const size_t n = (size_t)w * h;
    const int xc = min(x, (int)w - 1);
    bool in_x[5];
    int at_x[5];
#pragma unroll
    for (int c = 0; c < 5; ++c) {
        const int sx = x + (c - 2) * step;
        in_x[c] = sx >= 0 && sx < (int)w;
        at_x[c] = min(max(sx, 0), (int)w - 1);
    }
    const float e0 = strengths.x * -LOG2E, e1 = strengths.y * -LOG2E, e2 = strengths.z * -LOG2E, e3 = strengths.w * -LOG2E;
    V3 centre[ROWS], cn[ROWS], ca[ROWS], sum[ROWS];
    float cd[ROWS], lc[ROWS], inv_d[ROWS], inv_l[ROWS], inv_n[ROWS], weight[ROWS];
#pragma unroll
    for (int k = 0; k < ROWS; ++k) {
        const int y = min(y0 + k * step, (int)h - 1);
        const size_t i = (size_t)y * w + xc;
        centre[k] = load3(in + 3 * i);
        if constexpr (FIRST) {  // a firefly takes its neighbours' mean
            float near_top = 0.0f, near_n = 0.0f;
            V3 near_sum = v3(0, 0, 0);
            for (int dy = -1; dy <= 1; ++dy)
                for (int dx = -1; dx <= 1; ++dx) {
                    const int sx = xc + dx, sy = y + dy;
                    if ((dx == 0 && dy == 0) || sx < 0 || sy < 0 || sx >= (int)w || sy >= (int)h) continue;
                    const V3 c = load3(in + 3 * ((size_t)sy * w + sx));
                    near_top = fmax_(near_top, luma_of(c));
                    near_sum = near_sum + c;
                    near_n = near_n + 1.0f;
                }
            if (near_n > 0.0f && luma_of(centre[k]) > 1.5f * near_top + 0.05f) centre[k] = near_sum / near_n;
        }
        const float4 fa = feat[2 * i], fb = feat[2 * i + 1];
        ca[k] = v3(fa.x, fa.y, fa.z);
        cn[k] = v3(fb.x, fb.y, fb.z);
        cd[k] = fa.w;
        inv_n[k] = fb.w;
        lc[k] = luma_of(centre[k]);
        inv_d[k] = 1.0f / fmax_(fabsf(cd[k]), 1e-3f);
        inv_l[k] = 1.0f / (0.08f + lc[k]);
        sum[k] = v3(0, 0, 0);
        weight[k] = 0.0f;
    }
    constexpr float KERNEL[3] = {0.375f, 0.25f, 0.0625f};
#pragma unroll
    for (int r = -2; r < ROWS + 2; ++r) {
        const int sy = y0 + r * step;
        if (sy < 0 || sy >= (int)h) continue;
        const size_t row = (size_t)sy * w;
#pragma unroll
        for (int c = 0; c < 5; ++c) {
            const size_t j = row + (size_t)at_x[c];
            const float4 fa = feat[2 * j], fb = feat[2 * j + 1];
            const V3 raw = load3(in + 3 * j);
            const float raw_l = luma_of(raw);
            if (!in_x[c]) continue;
#pragma unroll
            for (int k = 0; k < ROWS; ++k) {
                const int dy = r - k;
                if (dy < -2 || dy > 2) continue;
                if ((fa.w < 0.0f) != (cd[k] < 0.0f)) continue;
                const bool own = dy == 0 && c == 2;
                const V3 tap = own ? centre[k] : raw;
                const float dn = fmax_(0.0f, 1.0f - dotf(cn[k], v3(fb.x, fb.y, fb.z)));
                const V3 dav = v3(fa.x, fa.y, fa.z) - ca[k];
                const float da = __builtin_amdgcn_sqrtf(dotf(dav, dav));
                const float dd = fabsf(fa.w - cd[k]) * inv_d[k];
                const float dl = fabsf((own ? lc[k] : raw_l) - lc[k]) * inv_l[k];
                float e = __builtin_fmaf(dn, e0, __builtin_fmaf(da, e1, __builtin_fmaf(dd, e2, dl * dl * e3)));
                e = e < -126.f ? -126.f : e;
                const float m = KERNEL[dy < 0 ? -dy : dy] * KERNEL[c < 2 ? 2 - c : c - 2] * __builtin_amdgcn_exp2f(e);
                sum[k] = v3(__builtin_fmaf(tap.x, m, sum[k].x), __builtin_fmaf(tap.y, m, sum[k].y), __builtin_fmaf(tap.z, m, sum[k].z));
                weight[k] = weight[k] + m;
            }
        }
    }
    if (x >= (int)w) return;
#pragma unroll
    for (int k = 0; k < ROWS; ++k) {
        const int y = y0 + k * step;
        if (y >= (int)h) return;
        const size_t i = (size_t)y * w + x;
        const V3 o = weight[k] > 0.0f ? sum[k] / weight[k] : centre[k];
        if constexpr (!LAST) store3(out + 3 * i, o);
        else finish_pixel(px, n, i, o, ca[k], inv_n[k], keep, view);
    }
}

// Pass `round` of the four over a w x h image by the table (feat, col0).
template <int ROWS>
void atrous_pass(phr_gpu* g, uint32_t* px, uint32_t w, uint32_t h, uint32_t round, uint32_t keep, const float s[4], float4 view,
                 const float4* feat, const float* col0) {
    const size_t n = (size_t)w * h;
    const uint32_t step = 1u << round, sets = (h + ROWS * step - 1) / (ROWS * step) * step;
    const dim3 grid((w + 63) / 64, (sets + 3) / 4), block(256);
    float* p14 = (float*)px + 14 * n;
    float* p17 = (float*)px + 17 * n;
    const float4 st = make_float4(s[0], s[1], s[2], s[3]);
    if (round == 0u)
        hipLaunchKernelGGL((k_atrous<ROWS, true, false>), grid, block, 0, g->stream, px, w, h, round, keep, st, view, feat, col0, p14);
    else if (round == 3u)
        hipLaunchKernelGGL((k_atrous<ROWS, false, true>), grid, block, 0, g->stream, px, w, h, round, keep, st, view, feat, p14, nullptr);
    else
        hipLaunchKernelGGL((k_atrous<ROWS, false, false>), grid, block, 0, g->stream, px, w, h, round, keep, st, view, feat,
                           round == 1u ? p14 : p17, round == 1u ? p17 : p14);
}

}  // namespace

// One pass (the `denoise` kernel of a recorded Pass).
int phr_denoise_pass_enqueue(phr_gpu* g, uint32_t* px, uint32_t w, uint32_t h, uint32_t step, uint32_t round, uint32_t last,
                             uint32_t keep, const float s[4], const float view[4]) {
    const size_t n = (size_t)w * h;
    if (n == 0) return PHR_OK;
    hipLaunchKernelGGL(k_denoise, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, g->stream, px, w, h, step, round, last,
                       keep, s[0], s[1], s[2], s[3], make_float4(view[0], view[1], view[2], view[3]));
    PHR_HIP(hipGetLastError());
    return PHR_OK;
}

// Enqueue the four passes of Tracer::denoise_with over an image buffer of w x h.
// With `scratch` (DENOISE_SCRATCH_WORDS words a pixel, 16-B aligned) the
// guides are derived once into it; without, every pass derives them again.
// view: the camera's colour-management words (transform 0, exposure, gamma).
int phr_denoise_enqueue(phr_gpu* g, uint32_t* px, uint32_t w, uint32_t h, int keep, float* scratch, const float view[4]) {
    const float s[4] = {64.0f, 8.0f, 40.0f, 7.0f};
    const uint32_t steps[4] = {1, 2, 4, 8};
    const size_t n = (size_t)w * h;
    if (n == 0) return PHR_OK;
    const dim3 grid((uint32_t)((n + 255) / 256));
    if (scratch) {
        float4* feat = (float4*)scratch;
        float* col0 = scratch + 8 * n;
        hipLaunchKernelGGL(k_denoise_prep, grid, dim3(256), 0, g->stream, (const uint32_t*)px, n, feat, col0);
        const float4 v4 = make_float4(view[0], view[1], view[2], view[3]);
        for (uint32_t r = 0; r < 4; ++r) {
            if (n >= ROWS3_MIN) atrous_pass<3>(g, px, w, h, r, keep ? 1u : 0u, s, v4, feat, col0);
            else if (n >= ROWS2_MIN) atrous_pass<2>(g, px, w, h, r, keep ? 1u : 0u, s, v4, feat, col0);
            else atrous_pass<1>(g, px, w, h, r, keep ? 1u : 0u, s, v4, feat, col0);
        }
    } else {
        for (uint32_t r = 0; r < 4; ++r)
            hipLaunchKernelGGL(k_denoise, grid, dim3(256), 0, g->stream, px, w, h, steps[r], r, steps[r] == 8 ? 1u : 0u,
                               keep ? 1u : 0u, s[0], s[1], s[2], s[3], make_float4(view[0], view[1], view[2], view[3]));
    }
    PHR_HIP(hipGetLastError());
    return PHR_OK;
}
