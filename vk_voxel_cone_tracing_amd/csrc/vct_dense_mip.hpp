// vct_dense_mip.hpp - one destination texel of the dense grid's anisotropic
// mip (radianceDownSample.comp:95-139 without the clipmap transition band),
// shared by vct_dense_mipmap and the batched launch so both run the same
// arithmetic.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "vct_internal.hpp"
#include "vct_texel.hpp"

namespace vct {

template <bool kF32>
__device__ __forceinline__ f4 dense_load(const void* base, size_t i)
{
    if (kF32) {
        const float4 t = ((const float4*)base)[i];
        return {t.x, t.y, t.z, t.w};
    }
    return unpack_unorm(((const uint32_t*)base)[i]);
}

template <bool kF32>
__device__ __forceinline__ void dense_store(void* base, size_t i, f4 v)
{
    if (kF32) ((float4*)base)[i] = make_float4(v.x, v.y, v.z, v.w);
    else ((uint32_t*)base)[i] = pack_unorm(v);
}

// The face-f value of a parent from its 8 children: the mean of 4 front-to-back
// pairs a + (1 - a.alpha) * b, accumulated in pair order.
__device__ __forceinline__ f4 dense_mip_face(const f4 v[8], int f)  // f must unroll to a constant
{
#pragma clang fp contract(off)
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const f4 a = v[face_pair_child(f, p, 0)];
        const f4 b = v[face_pair_child(f, p, 1)];
        const float t = 1.0f - a.w;
        acc[0] = acc[0] + a.x;
        acc[0] = acc[0] + t * b.x;
        acc[1] = acc[1] + a.y;
        acc[1] = acc[1] + t * b.y;
        acc[2] = acc[2] + a.z;
        acc[2] = acc[2] + t * b.z;
        acc[3] = acc[3] + a.w;
        acc[3] = acc[3] + t * b.w;
    }
    return f4{acc[0] * 0.25f, acc[1] * 0.25f, acc[2] * 0.25f, acc[3] * 0.25f};
}

// The packed texels i and i + 1 of a bordered RGBA8 block as one 8-byte load
// (4-byte aligned: interior pairs start at odd indices).
struct __attribute__((packed, aligned(4))) TexelPair {
    uint32_t a, b;
};

// The 8 children of destination texel (x, y, z) from face `src` of the level
// below, (2n)^3 interior texels.
template <bool kF32>
__device__ __forceinline__ void dense_mip_children(const void* __restrict__ src, int n, int x, int y, int z, f4 v[8])
{
    const size_t Ds = (size_t)(2 * n) + 2;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const size_t i = ((size_t)(2 * z + (r >> 1) + 1) * Ds + (size_t)(2 * y + (r & 1) + 1)) * Ds + (size_t)(2 * x + 1);
        if (kF32) {
            v[2 * r] = dense_load<true>(src, i);
            v[2 * r + 1] = dense_load<true>(src, i + 1);
        } else {
            const TexelPair t = *(const TexelPair*)((const uint32_t*)src + i);
            v[2 * r] = unpack_unorm(t.a);
            v[2 * r + 1] = unpack_unorm(t.b);
        }
    }
}

__device__ __forceinline__ size_t dense_mip_index(int n, int x, int y, int z)
{
    const size_t D = (size_t)n + 2;
    return ((size_t)(z + 1) * D + (size_t)(y + 1)) * D + (size_t)(x + 1);
}

__device__ __forceinline__ size_t dense_mip_block(int n)
{
    const size_t D = (size_t)n + 2;
    return D * D * D;
}

// The six faces of destination texel (x, y, z) of the level above level 0,
// which has one face: its 8 children are read and decoded once.
template <bool kF32>
__device__ __forceinline__ void dense_mip_first(const void* __restrict__ src, void* __restrict__ dst, int n, int x,
                                                int y, int z)
{
    f4 v[8];
    dense_mip_children<kF32>(src, n, x, y, z, v);
    const size_t di = dense_mip_index(n, x, y, z), dblock = dense_mip_block(n);
#pragma unroll
    for (int f = 0; f < kFaces; ++f) dense_store<kF32>(dst, (size_t)f * dblock + di, dense_mip_face(v, f));
}

// dense_mip_face for a face that is not a compile-time constant (uniform in
// the wave).
__device__ __forceinline__ f4 dense_mip_any_face(const f4 v[8], int f)
{
    switch (f) {
    case 0: return dense_mip_face(v, 0);
    case 1: return dense_mip_face(v, 1);
    case 2: return dense_mip_face(v, 2);
    case 3: return dense_mip_face(v, 3);
    case 4: return dense_mip_face(v, 4);
    default: return dense_mip_face(v, 5);
    }
}

// Destination texel (x, y, z) of face f of a level with n^3 interior texels
// from face f of the level below.
template <bool kF32>
__device__ __forceinline__ void dense_mip_texel(const void* __restrict__ src, void* __restrict__ dst, int n, int x,
                                                int y, int z, int f)
{
    f4 v[8];
    const size_t texel = kF32 ? 16 : 4;
    dense_mip_children<kF32>((const char*)src + (size_t)f * dense_mip_block(2 * n) * texel, n, x, y, z, v);
    dense_store<kF32>(dst, (size_t)f * dense_mip_block(n) + dense_mip_index(n, x, y, z), dense_mip_any_face(v, f));
}

// The last levels of a pyramid in one launch: the faces are independent from
// level 1 on, so one workgroup per face takes every level of at most kTailEdge
// texels an edge, each read from the one before in LDS. A launch for each of
// these levels costs 5 to 9 us for a few hundred texels (256^3 RGBA8: five
// launches, 41 us, are one of 14).
constexpr int kTailEdge8 = 16, kTailEdge32 = 8;  // RGBA8 / RGBA32F: 16 KB and 8 KB for the largest level

template <bool kF32>
constexpr int tail_edge()
{
    return kF32 ? kTailEdge32 : kTailEdge8;
}

template <bool kF32>
constexpr int tail_texels()  // the tail's levels that another level is made from: all but the last, 1^3
{
    int texels = 0;
    for (int e = tail_edge<kF32>(); e > 1; e /= 2) texels += e * e * e;
    return texels;
}

// Face f of levels m, m + 1, ..., nlevels - 1 (res >> m <= tail_edge), level l
// starting at texel offset[l] of `data`. Every thread of the workgroup calls it.
template <bool kF32>
__device__ __forceinline__ void dense_mip_tail(void* data, const unsigned long long* offset, int res, int m, int nlevels,
                                               int f)
{
    using T = typename std::conditional<kF32, float4, uint32_t>::type;
    __shared__ T lds[tail_texels<kF32>()];
    const T* below = nullptr;  // the level below in LDS, unbordered
    T* here = lds;
    for (; m < nlevels; ++m) {
        const int n = res >> m, sh = __builtin_ctz((unsigned)n);
        T* dst = (T*)data + offset[m] + (size_t)f * dense_mip_block(n);
        const T* src = (const T*)data + offset[m - 1] + (m == 1 ? 0 : (size_t)f * dense_mip_block(2 * n));
        for (int i = threadIdx.x; i < n * n * n; i += blockDim.x) {
            const int x = i & (n - 1), y = (i >> sh) & (n - 1), z = i >> (2 * sh);
            f4 v[8];
            if (below) {
#pragma unroll
                for (int c = 0; c < 8; ++c)
                    v[c] = dense_load<kF32>(below, (size_t)(((2 * z + (c >> 2)) * 2 * n + 2 * y + ((c >> 1) & 1)) * 2 * n +
                                                            2 * x + (c & 1)));
            } else {
                dense_mip_children<kF32>(src, n, x, y, z, v);
            }
            const f4 o = dense_mip_any_face(v, f);
            dense_store<kF32>(dst, dense_mip_index(n, x, y, z), o);
            if (m + 1 < nlevels) dense_store<kF32>(here, (size_t)i, o);
        }
        __syncthreads();
        below = here;
        here += n * n * n;
    }
}

// The arithmetic of one destination texel with one face at a time (the face
// loop is not unrolled and each pair's children are loaded by computed index),
// for kernels that must keep few registers live: the persistent batched launch,
// whose pixel tiles would otherwise inherit the unrolled version's registers.
template <bool kF32>
__device__ __forceinline__ void dense_mip_texel_lean(const void* src, void* dst, int n, int x, int y, int z,
                                                     bool src_single_face)
{
#pragma clang fp contract(off)
    const size_t Ds = (size_t)(2 * n) + 2, Dd = (size_t)n + 2;
    const size_t sblock = Ds * Ds * Ds, dblock = Dd * Dd * Dd;
    auto child = [&](size_t sface, int i) {
        return sface + ((size_t)(2 * z + (i >> 2) + 1) * Ds + (size_t)(2 * y + ((i >> 1) & 1) + 1)) * Ds +
               (size_t)(2 * x + (i & 1) + 1);
    };
#pragma unroll 1
    for (int f = 0; f < kFaces; ++f) {
        const size_t sface = src_single_face ? 0 : (size_t)f * sblock;
        float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const f4 a = dense_load<kF32>(src, child(sface, face_pair_child(f, p, 0)));
            const f4 b = dense_load<kF32>(src, child(sface, face_pair_child(f, p, 1)));
            const float t = 1.0f - a.w;
            acc[0] = acc[0] + a.x;
            acc[0] = acc[0] + t * b.x;
            acc[1] = acc[1] + a.y;
            acc[1] = acc[1] + t * b.y;
            acc[2] = acc[2] + a.z;
            acc[2] = acc[2] + t * b.z;
            acc[3] = acc[3] + a.w;
            acc[3] = acc[3] + t * b.w;
        }
        const size_t di = (size_t)f * dblock + ((size_t)(z + 1) * Dd + (size_t)(y + 1)) * Dd + (size_t)(x + 1);
        dense_store<kF32>(dst, di, f4{acc[0] * 0.25f, acc[1] * 0.25f, acc[2] * 0.25f, acc[3] * 0.25f});
    }
}

}  // namespace vct
