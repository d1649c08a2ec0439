// vct_filter.hip - the step after the cone trace: SpecularFilterPass
// (specularFilter.frag:25-53). Per pixel: the traced diffuse contribution plus
// the specular contribution filtered by the 32-direction x 8-ring blur
// (filter.glsl:9-24) or the 15x15 bilateral filter (filter.glsl:26-63), then
// the optional Uncharted2 tonemap (tonemapping.glsl:9-26). Inputs are sampled
// like the reference's "VCTSampler": bilinear, clamp to edge. Workgroups run in
// XCD order; the inputs are the two RGBA32F images the trace wrote.
#include <hip/hip_runtime.h>

#include <cmath>

#include "vct_internal.hpp"

static_assert(sizeof(vct_specular_filter_desc) == 16, "SpecularFilterPassDesc layout");

namespace vct {

__device__ __forceinline__ float4 tex_clamp_linear(const float4* __restrict__ img, int W, int H, float s, float t)
{
#pragma clang fp contract(off)
    const float u = s * (float)W - 0.5f, v = t * (float)H - 0.5f;
    const float fu = floorf(u), fv = floorf(v);
    const float a = u - fu, b = v - fv;
    const int i0 = (int)fu, j0 = (int)fv;
    float4 r = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
    for (int dy = 0; dy < 2; ++dy)
#pragma unroll
        for (int dx = 0; dx < 2; ++dx) {
            int i = i0 + dx, j = j0 + dy;
            i = i < 0 ? 0 : (i > W - 1 ? W - 1 : i);
            j = j < 0 ? 0 : (j > H - 1 ? H - 1 : j);
            const float w = (dx ? a : 1.0f - a) * (dy ? b : 1.0f - b);
            const float4 p = img[(size_t)j * (size_t)W + (size_t)i];
            r.x += w * p.x;
            r.y += w * p.y;
            r.z += w * p.z;
            r.w += w * p.w;
        }
    return r;
}

// The bilateral filter's 15 spatial weights, |offset| 0..7.
__constant__ float c_kernel8[8] = {0.039894000f, 0.039695028f, 0.039104044f, 0.038138565f,
                                   0.036826804f, 0.035206333f, 0.033322271f, 0.031225216f};

__host__ __device__ __forceinline__ float uncharted2(float x)
{
#pragma clang fp contract(off)
    const float A = 0.15f, B = 0.50f, C = 0.10f, D = 0.20f, E = 0.02f, F = 0.30f;
    return ((x * (A * x + C * B) + D * E) / (x * (A * x + B) + D * F)) - E / F;
}

// The tonemap's constants, the same for every pixel.
struct Tonemap {
    int enable;
    float exposure;
    float white;      // 1 / uncharted2(11.2)
    float inv_gamma;
};

__device__ __forceinline__ float4 combine(float4 col, float sx, float sy, float sz, const Tonemap& T)
{
#pragma clang fp contract(off)
    col.x += sx;
    col.y += sy;
    col.z += sz;
    if (T.enable)
        col = make_float4(powf(uncharted2(col.x * T.exposure) * T.white, T.inv_gamma),
                          powf(uncharted2(col.y * T.exposure) * T.white, T.inv_gamma),
                          powf(uncharted2(col.z * T.exposure) * T.white, T.inv_gamma), col.w);
    return col;
}

// filter.glsl:9-24. The blur's rings are 0.01 / size wide in texture
// coordinates: every one of its 256 taps lies within 0.01 texel of the pixel's
// centre, so its bilinear footprint stays in the 3x3 texels around the pixel
// and the sum of all taps is a 3x3 stencil whose weights are the same for
// every pixel and image. The host sums them in double precision (blur_stencil).
// The stencil sits on the texel's centre itself: an FP32 texture coordinate
// would miss it by up to 6e-5 texel at 1920, the larger part of the error of
// taps evaluated one by one (1920x1080 without the tonemap: 1.9e-6 of the
// image's norm against 64 bits, now 6e-7).
struct BlurStencil {
    float w[3][3];
};

// Bound by HBM (two images read, one written), with the tonemap by its three
// powers a pixel. One lane per pixel, 64 x 4 pixels per workgroup, so a wave
// reads and writes whole 1 KB row pieces; the 3x3 neighbours come from the L1.
// 1920x1080: 943 us (with tonemap) with the 256 taps evaluated one by one, about
// 1000 texel loads a pixel; now 17 us, 34 with the tonemap's powers (100 MB, 5.9
// and 2.9 TB/s).
__global__ __launch_bounds__(256) void k_specular_blur(const float4* __restrict__ diffuse,
                                                       const float4* __restrict__ specular, int W, int H,
                                                       BlurStencil S, Tonemap T, float4* __restrict__ out)
{
    const unsigned tiles_x = ((unsigned)W + 63u) / 64u;
    const unsigned tile = xcd_remap(blockIdx.x, gridDim.x);
    const int px = (int)(tile % tiles_x) * 64 + (int)(threadIdx.x & 63);
    const int py = (int)(tile / tiles_x) * 4 + (int)(threadIdx.x >> 6);
    if (px >= W || py >= H) return;
    const int xs[3] = {px > 0 ? px - 1 : 0, px, px < W - 1 ? px + 1 : px};
    const int ys[3] = {py > 0 ? py - 1 : 0, py, py < H - 1 ? py + 1 : py};
    float ax = 0.0f, ay = 0.0f, az = 0.0f;
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const float4 q = specular[(size_t)ys[j] * (size_t)W + (size_t)xs[i]];
            const float w = S.w[j][i];
            ax += w * q.x;
            ay += w * q.y;
            az += w * q.z;
        }
    const float4 col = tex_clamp_linear(diffuse, W, H, ((float)px + 0.5f) / (float)W, ((float)py + 0.5f) / (float)H);
    out[(size_t)py * (size_t)W + (size_t)px] = combine(col, ax, ay, az, T);
}

// filter.glsl:26-63. The 15 x 15 taps lie on texel centres, so each is one
// texel (clamped to the edge): the tile's texels and their 7-texel halo are
// staged in LDS once, 64 x (4 * kRows) pixels per workgroup, and a lane takes
// kRows pixels of one column, so one LDS read serves up to kRows of them.
// Bound by the vector ALU: 225 weights (one hardware exp2 each) per pixel.
// 1919x1077: 177 us, 199 with the tonemap.
// 1/(2 sigma^2) with sigma = 10; the Gaussian's normalisation cancels in the
// quotient.
template <int kRows>
__global__ __launch_bounds__(256) void k_specular_bilateral(const float4* __restrict__ diffuse,
                                                            const float4* __restrict__ specular, int W, int H,
                                                            Tonemap T, float4* __restrict__ out)
{
    constexpr int R = 7, TW = 64 + 2 * R, TH = 4 * kRows + 2 * R;
    __shared__ float4 tex[TH * TW];
    const unsigned tiles_x = ((unsigned)W + 63u) / 64u;
    const unsigned tile = xcd_remap(blockIdx.x, gridDim.x);
    const int x0 = (int)(tile % tiles_x) * 64, y0 = (int)(tile / tiles_x) * (4 * kRows);
    for (int k = threadIdx.x; k < TH * TW; k += 256) {
        const int x = x0 + k % TW - R, y = y0 + k / TW - R;
        const int cx = x < 0 ? 0 : (x > W - 1 ? W - 1 : x), cy = y < 0 ? 0 : (y > H - 1 ? H - 1 : y);
        tex[k] = specular[(size_t)cy * (size_t)W + (size_t)cx];
    }
    __syncthreads();
    const int lx = (int)(threadIdx.x & 63), ly = (int)(threadIdx.x >> 6) * kRows;
    float4 c[kRows];
    float Z[kRows], ax[kRows], ay[kRows], az[kRows];
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        c[r] = tex[(ly + r + R) * TW + lx + R];
        Z[r] = ax[r] = ay[r] = az[r] = 0.0f;
    }
    const float e = -0.5f / 100.0f * 1.44269504f;  // exp(x) = exp2(x log2(e))
#pragma unroll 1
    for (int i = -R; i <= R; ++i) {
        const float ki = c_kernel8[i < 0 ? -i : i];
#pragma unroll
        for (int j = 0; j < kRows + 2 * R; ++j) {
            const float4 q = tex[(ly + j) * TW + lx + R + i];
#pragma unroll
            for (int r = 0; r < kRows; ++r) {
                const int dj = j - r - R;
                if (dj < -R || dj > R) continue;
                const float dx = q.x - c[r].x, dy = q.y - c[r].y, dz = q.z - c[r].z;
                const float dd = dx * dx + dy * dy + dz * dz;
                const float f = __builtin_amdgcn_exp2f(dd * e) * (ki * c_kernel8[dj < 0 ? -dj : dj]);
                Z[r] += f;
                ax[r] += f * q.x;
                ay[r] += f * q.y;
                az[r] += f * q.z;
            }
        }
    }
    const int px = x0 + lx;
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        const int py = y0 + ly + r;
        if (px >= W || py >= H) continue;
        const float4 col =
            tex_clamp_linear(diffuse, W, H, ((float)px + 0.5f) / (float)W, ((float)py + 0.5f) / (float)H);
        out[(size_t)py * (size_t)W + (size_t)px] = combine(col, ax[r] / Z[r], ay[r] / Z[r], az[r] / Z[r], T);
    }
}

// Workgroups of 64 x 16 pixels from which the four-row bilateral kernel is
// used: two for each of the 256 CUs, and a wave there runs four times as long
// as with one row. Smaller images are cut four times finer (640x360: 32 us,
// 160x90: 13 us).
constexpr unsigned kBilateralTallTiles = 512;

// The blur's taps (the shader's float loops over 32 directions and 8 rings,
// and the centre tap) as one stencil over the quotient 8 * 32 - 15.
static BlurStencil blur_stencil()
{
    double w[3][3] = {};
    auto add = [&](double dx, double dy) {
        const double wx[3] = {dx < 0 ? -dx : 0.0, 1.0 - std::fabs(dx), dx > 0 ? dx : 0.0};
        const double wy[3] = {dy < 0 ? -dy : 0.0, 1.0 - std::fabs(dy), dy > 0 ? dy : 0.0};
        for (int j = 0; j < 3; ++j)
            for (int i = 0; i < 3; ++i) w[j][i] += wy[j] * wx[i];
    };
    add(0.0, 0.0);
    const float two_pi = 6.28318530718f;
    for (float a = 0.0f; a < two_pi; a += two_pi / 32.0f)
        for (float i = 1.0f / 8.0f; i <= 1.0f; i += 1.0f / 8.0f)
            add((double)std::cos(a) * 0.01 * i, (double)std::sin(a) * 0.01 * i);
    const double n = 8.0 * 32.0 - 15.0;
    BlurStencil S;
    for (int j = 0; j < 3; ++j)
        for (int i = 0; i < 3; ++i) S.w[j][i] = (float)(w[j][i] / n);
    return S;
}

}  // namespace vct

using namespace vct;

extern "C" vct_status vct_specular_filter(vct_stream stream, const float* diffuse, const float* specular, uint32_t width,
                                          uint32_t height, const vct_specular_filter_desc* desc, float* out)
{
    if (!diffuse || !specular || !desc || !out || !width || !height)
        return fail(VCT_ERR_INVALID_ARGUMENT, "null argument or empty image");
    if (out == diffuse || out == specular) return fail(VCT_ERR_INVALID_ARGUMENT, "out must not alias an input");
    hipStream_t s = (hipStream_t)stream;
    const int W = (int)width, H = (int)height;
    const float4 *d = (const float4*)diffuse, *sp = (const float4*)specular;
    const Tonemap T{desc->tonemap_enable == 1, desc->tonemap_exposure, 1.0f / uncharted2(11.2f),
                    1.0f / desc->tonemap_gamma};
    const unsigned cols = (width + 63) / 64;
    if (desc->filter_method == 1) {
        static const BlurStencil S = blur_stencil();
        hipLaunchKernelGGL(k_specular_blur, dim3(cols * ((height + 3) / 4)), dim3(256), 0, s, d, sp, W, H, S, T,
                           (float4*)out);
    } else if (cols * ((height + 15) / 16) >= kBilateralTallTiles) {
        hipLaunchKernelGGL(k_specular_bilateral<4>, dim3(cols * ((height + 15) / 16)), dim3(256), 0, s, d, sp, W, H, T,
                           (float4*)out);
    } else {
        hipLaunchKernelGGL(k_specular_bilateral<1>, dim3(cols * ((height + 3) / 4)), dim3(256), 0, s, d, sp, W, H, T,
                           (float4*)out);
    }
    VCT_HIP(hipGetLastError());
    return VCT_OK;
}
