// vct_expand.hpp - the expansion of triangles into work items, shared by the
// voxelizers. The items of triangle t (its raster samples) are numbered from
// the exclusive prefix of the triangles' counts. The prefix is kept in two
// parts: within the triangle's block of 256, written by the kernel that
// counts (expand_block), and of the blocks, scanned by one workgroup
// (expand_scan); a separate scan pass over the triangles would read and write
// them again in launches of its own.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace vct {

constexpr uint32_t kExpandBlock = 256;  // triangles per block: the counting kernels' workgroup

// Where each triangle's items begin: triangle t's are numbered from
// block[t / 256] + in_block[t].
struct Expansion {
    const unsigned long long* in_block;
    const unsigned long long* block;

    __device__ __forceinline__ unsigned long long operator()(uint32_t t) const
    {
        return block[t / kExpandBlock] + in_block[t];
    }
};

// Called by every thread of a 256-thread workgroup with its triangle's item
// count (0 past the last triangle): returns the sum of the lower threads'
// counts and leaves the workgroup's sum in *block_sum. Sums are 64 bits wide: 256
// triangles of millions of samples each pass 2^32.
__device__ __forceinline__ unsigned long long expand_block(unsigned long long count, unsigned long long* block_sum)
{
    __shared__ unsigned long long wave_sum[kExpandBlock / 64];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    unsigned long long v = count;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const unsigned long long u = __shfl_up(v, off, 64);
        if (lane >= (uint32_t)off) v += u;
    }
    if (lane == 63u) wave_sum[wave] = v;
    __syncthreads();
    unsigned long long below = 0, all = 0;
#pragma unroll
    for (uint32_t w = 0; w < kExpandBlock / 64; ++w) {
        if (w < wave) below += wave_sum[w];
        all += wave_sum[w];
    }
    if (threadIdx.x == 0) *block_sum = all;
    return below + v - count;
}

// Exclusive prefix of sums[0, n) in place, by one workgroup of 1024 threads
// (each a contiguous run); returns the total to every thread. Serial in n / 1024,
// and no slower than the library scan of all the triangles' counts (256 n of 8
// bytes) that it stands for until n is beyond any draw list: 7 us for 4096 sums
// (1M triangles), 47 for 27 800 (7.1M), 427 for 262 144 (67M), against 21, 65 and
// 415 us; a scan of 1024 n flags, which k_svo_cover's counts replace, took 31, 109
// and 811 us.
__device__ __forceinline__ unsigned long long expand_scan(unsigned long long* sums, uint32_t n)
{
    __shared__ unsigned long long wave_sum[16];
    const uint32_t per = (n + 1023u) / 1024u, lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t lo = min(threadIdx.x * per, n), hi = min(lo + per, n);
    unsigned long long own = 0;
    for (uint32_t i = lo; i < hi; ++i) own += sums[i];
    unsigned long long v = own;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const unsigned long long u = __shfl_up(v, off, 64);
        if (lane >= (uint32_t)off) v += u;
    }
    if (lane == 63u) wave_sum[wave] = v;
    __syncthreads();
    unsigned long long below = 0, all = 0;
#pragma unroll
    for (uint32_t w = 0; w < 16u; ++w) {
        if (w < wave) below += wave_sum[w];
        all += wave_sum[w];
    }
    unsigned long long run = below + v - own;
    for (uint32_t i = lo; i < hi; ++i) {
        const unsigned long long s = sums[i];
        sums[i] = run;
        run += s;
    }
    return all;
}

// The triangle of each lane's work item, the wave's items being consecutive:
// item first + lane, lanes past `last` taking item last. at(t) is where the
// items of triangle t in [0, n) begin (nondecreasing; n >= 1, at(0) <= first
// and every item of the wave belongs to a triangle below n): the answer is the
// last t with at(t) <= item. The whole wave must call it. The wave's first
// triangle comes from a 64-way search (three dependent reads for 2^18
// triangles, not eighteen; the opacity raster of six 128^3 levels took 37 us for
// 44 with it); the lanes then search the next 64 starts, held one per lane, and
// only lanes past those search memory by themselves (where most triangles have
// no items).
template <typename At>
__device__ __forceinline__ uint32_t wave_triangle(const At& at, uint32_t n, unsigned long long first,
                                                  unsigned long long last)
{
    const uint32_t lane = threadIdx.x & 63u;
    const unsigned long long item = first + lane < last ? first + lane : last;
    uint32_t lo = 0, hi = n;  // the last start at or before `first` lies in [lo, hi)
    while (hi - lo > 1u) {
        const uint32_t step = (hi - lo + 63u) / 64u;
        const uint32_t t = lo + lane * step;
        const unsigned long long m = __ballot(t < hi && at(t) <= first);  // a prefix of the lanes, lane 0 among them
        const uint32_t k = 63u - (uint32_t)__clzll((long long)m);
        lo = lo + k * step;
        hi = min(lo + step, hi);
    }
    // starts lo + 1 + lane; past the last triangle nothing begins
    const uint32_t next = lo + 1u + lane;
    const unsigned long long start = next < n ? at(next) : ~0ull;
    uint32_t a = 0;  // starts of the window at or before the lane's item
#pragma unroll
    for (uint32_t b = 32; b > 0u; b >>= 1) {
        const unsigned long long s = __shfl(start, (int)(a + b - 1u), 64);
        if (s <= item) a += b;
    }
    if (a == 63u && __shfl(start, 63, 64) <= item) a = 64u;
    uint32_t t = lo + a;
    if (a == 64u) {  // beyond the window
        uint32_t end = n;
        while (end - t > 1u) {
            const uint32_t mid = (t + end) >> 1;
            if (at(mid) <= item) t = mid; else end = mid;
        }
    }
    return t;
}

}  // namespace vct
