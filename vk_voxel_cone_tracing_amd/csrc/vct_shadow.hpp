// vct_shadow.hpp - shadow-map visibility (shadow.glsl:8-36) shared by the
// radiance injector and the SVO fragment voxelizer. FP32 without contraction
// in the reference's operation order, so its result is reproducible bit for
// bit.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

#include "../../include/vct.h"

namespace vct {

struct LightParams {
    float dir[3];       // normalize(-direction)
    float color[3];
    float intensity;
    float view[16];
    float proj[16];
    float z_near, z_far;
    const float* depth;
    int width, height;
};

// A tap's first texel and weight along one axis.
__device__ __forceinline__ void tap_origin(float at, float size, int& first, float& frac)
{
#pragma clang fp contract(off)
    const float u = at * size - 0.5f, f = floorf(u);
    frac = u - f;
    first = (int)fminf(fmaxf(f, -4.0f), size + 4.0f);
}

// A texel as a tap weighs it: its depth, or how it compares.
__device__ __forceinline__ float tap_texel(const LightParams& L, int i, int j, bool compare, float ref)
{
    const bool in = i >= 0 && j >= 0 && i < L.width && j < L.height;  // CLAMP_TO_BORDER, opaque black
    const float t = in ? L.depth[(size_t)j * (size_t)L.width + (size_t)i] : 0.0f;
    return compare ? ((!in || ref <= t) ? 1.0f : 0.0f) : t;
}

__device__ __forceinline__ float tap_weigh(float a, float b, float t00, float t10, float t01, float t11)
{
#pragma clang fp contract(off)
    float r = ((1.0f - a) * (1.0f - b)) * t00;
    r = r + (a * (1.0f - b)) * t10;
    r = r + ((1.0f - a) * b) * t01;
    r = r + (a * b) * t11;
    return r;
}

// Five texels of one row of the window.
__device__ __forceinline__ void window_row(const LightParams& L, int i0, int j, bool compare, float ref, float row[5])
{
#pragma unroll
    for (int k = 0; k < 5; ++k) row[k] = tap_texel(L, i0 + k, j, compare, ref);
}

// shadow.glsl:28-36 calcVisibility + PCF16 (:14-26)
__device__ __forceinline__ float visibility(const LightParams& L, const float pos[3], uint32_t quirks)
{
#pragma clang fp contract(off)
    const float* V = L.view;
    const float* Pm = L.proj;
    float ls[3];
    for (int k = 0; k < 3; ++k) ls[k] = V[0 + k] * pos[0] + V[4 + k] * pos[1] + V[8 + k] * pos[2] + V[12 + k];
    const bool compare = !(quirks & VCT_QUIRK_SHADOW_RAW_DEPTH);
    float ref = 0.0f;
    if (compare) {
        ref = Pm[2] * ls[0] + Pm[6] * ls[1] + Pm[10] * ls[2] + Pm[14];
        ref = ref - 0.001f;
    }
    ls[2] = ls[2] / (L.z_far - L.z_near);
    float xy[2];
    for (int k = 0; k < 2; ++k) xy[k] = Pm[0 + k] * ls[0] + Pm[4 + k] * ls[1] + Pm[12 + k];
    xy[0] = xy[0] * 0.5f + 0.5f;
    xy[1] = xy[1] * 0.5f + 0.5f;
    const float sx = 1.0f / (float)L.width;
    const float sy = 1.0f / (float)L.height;
    // offsets -1.5, -0.5, 0.5, 1.5 (exact in float), y outer as in the
    // reference. The taps' columns depend on x alone and their rows on y alone,
    // and as a rule the four columns (rows) are consecutive: then all taps read
    // one window of 5 x 5 texels, each fetched and compared once (64 fetches
    // tap by tap). Where rounding or the border's clamp makes them other than
    // consecutive, the taps fetch for themselves. Bound by the fetches and
    // their bounds tests: octree fragments of 1M triangles at 2^9, shadow map
    // 2048^2, 694 -> 304 us; injection at 128^3 x 6 levels 68 -> 54 us.
    float fx[4], fy[4];
    int x0[4], y0[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float off = -1.5f + (float)k;
        tap_origin(xy[0] + off * sx, (float)L.width, x0[k], fx[k]);
        tap_origin(xy[1] + off * sy, (float)L.height, y0[k], fy[k]);
    }
    bool window = true;
#pragma unroll
    for (int k = 1; k < 4; ++k) window = window && x0[k] == x0[0] + k && y0[k] == y0[0] + k;
    if (window) {
        float sum = 0.0f, row[2][5];
        window_row(L, x0[0], y0[0], compare, ref, row[0]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            window_row(L, x0[0], y0[0] + j + 1, compare, ref, row[(j + 1) & 1]);
            const float* r0 = row[j & 1];
            const float* r1 = row[(j + 1) & 1];
#pragma unroll
            for (int i = 0; i < 4; ++i) sum = sum + tap_weigh(fx[i], fy[j], r0[i], r0[i + 1], r1[i], r1[i + 1]);
        }
        return sum * 0.0625f;
    }
    float sum = 0.0f;
#pragma unroll 1
    for (int j = 0; j < 4; ++j)
#pragma unroll 1
        for (int i = 0; i < 4; ++i) {
            int i0, j0;
            float a, b;
            tap_origin(xy[0] + (-1.5f + (float)i) * sx, (float)L.width, i0, a);
            tap_origin(xy[1] + (-1.5f + (float)j) * sy, (float)L.height, j0, b);
            sum = sum + tap_weigh(a, b, tap_texel(L, i0, j0, compare, ref), tap_texel(L, i0 + 1, j0, compare, ref),
                                  tap_texel(L, i0, j0 + 1, compare, ref), tap_texel(L, i0 + 1, j0 + 1, compare, ref));
        }
    return sum * 0.0625f;
}


}  // namespace vct
