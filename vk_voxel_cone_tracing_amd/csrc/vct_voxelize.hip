// vct_voxelize.hip - clip-level triangle voxelization (K1) and radiance
// injection (K2) for gfx950.
//
// Both passes take one or several clip levels per call and expand
// (level, triangle) pairs into (level, triangle, cell, sample) work items
// with one exclusive scan over the per-pair cell counts, so every wavefront
// gets an even share of raster work regardless of triangle size and level,
// and all levels of a pass share the launches (and, for K2, the one host
// wait for the record count and the one sort). K1 writes opacity
// directly (the stores are idempotent). K2 reproduces the reference's
// order-dependent imageAtomicCompSwap running average deterministically: each
// fragment emits one record per written face texel keyed by
// (texel address in the volume, work index), a radix sort groups the records
// by texel in fragment order (a texel belongs to one level, whose work items
// keep their order), and one lane per texel (a wave for a long run) applies the
// running average (RGBA8) or the FP32 sum/count mean (RGBA16F) in that order.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <cmath>
#include <cstring>

#include "vct_expand.hpp"
#include "vct_internal.hpp"
#include "vct_raster.hpp"
#include "vct_shadow.hpp"
#include "vct_texel.hpp"
#include "vct_textures.hpp"

namespace vct {

struct VoxParams {
    float region_min[3];
    float region_max[3];
    float clip_max_extent;
    float voxel_size;
    int clip_level;
    int res;
    int D;
    int lo[3];
    int hi[3];
    int samples;
    uint32_t quirks;
};

// Voxel cell of a coordinate on one axis: floor(p / voxel_size).
__device__ __forceinline__ int voxel_cell(const VoxParams& P, float p)
{
    return (int)floorf(p / P.voxel_size);
}

// msaaVoxelizer.frag:43-55 / msaaInjectRadiance.frag:162-174. With
// VCT_QUIRK_CLAMP_X_RANGE, the reference's calculateImageCoords: clamp into the
// closed region (with the x range on every axis), then fract(p / extent).
// Without it, half-open voxel cells: texel = cell mod res with the cell clamped
// into the region's cells, so a point's texel does not depend on where the
// region sits and a sub-region voxelization writes exactly the texels a full
// one writes inside it.
__device__ __forceinline__ void image_coords(const VoxParams& P, const float pos[3], int ic[3])
{
#pragma clang fp contract(off)
    if (P.quirks & VCT_QUIRK_CLAMP_X_RANGE) {
        const float c = P.voxel_size * 0.25f;
        for (int k = 0; k < 3; ++k) {
            const float lo = P.region_min[0] + c;
            const float hi = P.region_max[0] - c;
            const float w = fminf(fmaxf(pos[k], lo), hi);
            const float q = w / P.clip_max_extent;
            const float fr = q - floorf(q);
            ic[k] = ((int)(fr * (float)P.res)) % P.res + 1;
        }
        return;
    }
    for (int k = 0; k < 3; ++k) {
        const int g = min(max(voxel_cell(P, pos[k]), P.lo[k] + 1), P.hi[k] - 1);
        ic[k] = (g & (P.res - 1)) + 1;
    }
}

// msaaVoxelizer.frag:59-60: the reference keeps fragments in the closed region;
// without VCT_QUIRK_CLAMP_X_RANGE the region is its half-open cells.
__device__ __forceinline__ bool in_region(const VoxParams& P, const float fp[3])
{
    if (P.quirks & VCT_QUIRK_CLAMP_X_RANGE)
        return !(fp[0] < P.region_min[0] || fp[1] < P.region_min[1] || fp[2] < P.region_min[2] ||
                 fp[0] > P.region_max[0] || fp[1] > P.region_max[1] || fp[2] > P.region_max[2]);
    for (int k = 0; k < 3; ++k) {
        const int g = voxel_cell(P, fp[k]);
        if (g <= P.lo[k] || g >= P.hi[k]) return false;
    }
    return true;
}

// The clip levels of one call: their raster parameters and, for the
// injection, the depth-clip box of each. Passed by value (kernel arguments);
// a work item's slot is found from the slot starts the expansion wrote.
struct LevelSet {
    VoxParams P[kMaxLevels];
    float box_lo[kMaxLevels][3], box_hi[kMaxLevels][3];
    int n;               // slots in use
    uint32_t keep_mask;  // bit l: clip level l keeps its stored alpha (RGBA16F after vct_begin_radiance_level)
};

// The work items (cells x samples) of triangle t in the slot's level (grid:
// triangles x slots): their prefix within the block of 256 triangles, and the
// block's sum. With k_total this is the whole scan, 10 us in two launches (a
// library scan of the counts: 18 us in four).
__global__ __launch_bounds__(kExpandBlock) void k_count(const float* __restrict__ pos, uint32_t ntris, LevelSet S,
                                                        unsigned long long* __restrict__ in_block,
                                                        unsigned long long* __restrict__ block_sums)
{
    const uint32_t t = blockIdx.x * kExpandBlock + threadIdx.x, slot = blockIdx.y;
    unsigned long long n = 0;
    if (t < ntris) {
        const VoxParams& P = S.P[slot];
        float p[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) p[k] = pos[9u * t + k];
        TriSetup s;
        if (tri_setup(p, P.voxel_size, P.samples, P.lo, P.hi, s))
            n = (unsigned long long)s.nu * s.nv * (unsigned long long)P.samples;
    }
    const uint32_t b = slot * gridDim.x + blockIdx.x;
    const unsigned long long below = expand_block(n, &block_sums[b]);
    in_block[(size_t)b * kExpandBlock + threadIdx.x] = below;
}

// The work items of the slots are numbered consecutively, each slot starting
// at a multiple of 64 (kWaveAlign), so that every wave of a grid-stride loop
// (64 consecutive items from a multiple of 64) lies in one slot: the slot's
// parameters are then wave-uniform (scalar registers). totals layout:
// [0] the numbered items (padding included), [1] the injection's record
// counter (0), [2 + k] slot k's first item, [10 + k] its first item in the
// unpadded scan (offsets), [18 + k] its item count. The record counter
// (kTotRec) sits 256 bytes past the start, in a cache line of its own: every
// work item reads the slot table, and sharing a line with the counter that
// every fragment increments atomically would make each of those reads wait.
constexpr unsigned long long kWaveAlign = 64;
constexpr int kTotA = 2, kTotU = 2 + kMaxLevels, kTotC = 2 + 2 * kMaxLevels;
constexpr int kTotRec = 32, kTotWords = kTotRec + 1;
static_assert(kTotC + kMaxLevels <= kTotRec, "slot table overlaps the record counter");
static_assert(8u * kTotWords <= kPinnedWordBytes, "totals read back into the pinned landing slot");

// Scans the block sums (nblocks per slot) and writes the totals.
__global__ __launch_bounds__(1024) void k_total(unsigned long long* __restrict__ blocks, uint32_t nblocks, int nslots,
                                                unsigned long long* __restrict__ totals)
{
    const unsigned long long all = expand_scan(blocks, nblocks * (uint32_t)nslots);
    __syncthreads();
    if (threadIdx.x != 0) return;
    unsigned long long a = 0;
    for (int k = 0; k < nslots; ++k) {
        const unsigned long long u = nblocks ? blocks[(size_t)k * nblocks] : 0ull;
        const unsigned long long next = k + 1 < nslots && nblocks ? blocks[(size_t)(k + 1) * nblocks] : all;
        totals[kTotA + k] = a;
        totals[kTotU + k] = u;
        totals[kTotC + k] = next - u;
        a += (next - u + kWaveAlign - 1) / kWaveAlign * kWaveAlign;
    }
    totals[0] = a;
    totals[kTotRec] = 0ull;
}

__global__ void k_reset_records(unsigned long long* __restrict__ total) { total[kTotRec] = 0ull; }

// Bits of the work index in an injection record key: enough for n - 1 (n
// work items). The key is (texel index in the volume) << bits | index.
__host__ __device__ inline uint32_t work_bits(unsigned long long n)
{
    uint32_t b = 1;
    while (n > 1ull && b < 32 && ((n - 1ull) >> b) != 0ull) ++b;  // n <= 2^32 (checked)
    return b;
}

// The slot of work item wi (wave-uniform, see k_total), its position in the
// unpadded numbering (the work index the injection's record keys carry) and
// its triangle. The whole wave calls it with consecutive items from a multiple
// of 64. valid is false for a slot's padding.
struct WorkItem {
    int slot;
    bool valid;
    uint32_t t;       // triangle
    uint32_t sample;  // index of the (cell, sample) within the triangle
};

__device__ __forceinline__ WorkItem work_item(const Expansion& E, const unsigned long long* __restrict__ totals,
                                              uint32_t ntris, int nslots, unsigned long long wi)
{
    int slot = 0;
    for (int k = 1; k < nslots; ++k) slot += wi >= totals[kTotA + k] ? 1 : 0;
    slot = __builtin_amdgcn_readfirstlane(slot);  // one slot per wave
    WorkItem it;
    it.slot = slot;
    const unsigned long long local = wi - totals[kTotA + slot], count = totals[kTotC + slot], u = totals[kTotU + slot];
    it.valid = local < count;
    const uint32_t nblocks = (ntris + kExpandBlock - 1u) / kExpandBlock, base = (uint32_t)slot * nblocks;
    const Expansion slot_items{E.in_block + (size_t)base * kExpandBlock, E.block + base};
    const unsigned long long local0 = local - (threadIdx.x & 63u);  // a wave's first item is valid
    it.t = wave_triangle(slot_items, ntris, u + local0, u + count - 1ull);
    it.sample = it.valid ? (uint32_t)(u + local - slot_items(it.t)) : 0u;
    return it;
}

// The unpadded work index of item wi of `slot`.
__device__ __forceinline__ unsigned long long work_index(const unsigned long long* __restrict__ totals, int slot,
                                                         unsigned long long wi)
{
    return wi - totals[kTotA + slot] + totals[kTotU + slot];
}

__global__ __launch_bounds__(256) void k_raster_opacity(const float* __restrict__ pos,
                                                        Expansion E, uint32_t ntris,
                                                        const unsigned long long* __restrict__ totals, LevelSet S,
                                                        TexInputs T, uint32_t* __restrict__ vol)
{
    const unsigned long long n = totals[0];
    const unsigned long long stride = (unsigned long long)gridDim.x * blockDim.x;
    for (unsigned long long wi = (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x; wi < n; wi += stride) {
        const WorkItem it = work_item(E, totals, ntris, S.n, wi);
        if (!it.valid) continue;
        const VoxParams P = S.P[it.slot];
        const uint32_t t = it.t;
        float p[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) p[k] = pos[9u * t + k];
        TriSetup s;
        if (!tri_setup(p, P.voxel_size, P.samples, P.lo, P.hi, s)) continue;
        float fp[3];
        double lam[3];
        if (!tri_sample(p, s, P.voxel_size, P.samples, it.sample, fp, lam)) continue;
        if (!in_region(P, fp)) continue;
        if (T.tex) {
            // msaaVoxelizer.frag:64: occlusion-texture discard
            float uv[2];
            interp_uv(T.uv + 6u * t, lam, uv);
            if (occluded(T, T.mats[T.mat[t]], uv)) continue;
        }
        int ic[3];
        image_coords(P, fp, ic);
        // imageStore(vec4(1.0)) into the six faces (msaaVoxelizer.frag:69-73)
        for (int f = 0; f < kFaces; ++f) vol[vol_index(P.D, P.clip_level, f, ic[0], ic[1], ic[2])] = 0xffffffffu;
    }
}

struct Record {
    float r, g, b;
};

__global__ __launch_bounds__(256) void k_raster_inject(const float* __restrict__ pos, const float* __restrict__ nrm,
                                                       TexInputs T, Expansion E, uint32_t ntris,
                                                       unsigned long long* __restrict__ totals,
                                                       LevelSet S, LightParams L,
                                                       unsigned long long* __restrict__ keys,
                                                       uint32_t* __restrict__ idx, Record* __restrict__ vals,
                                                       uint32_t cap)
{
#pragma clang fp contract(off)
    __shared__ uint32_t wave_records[4];
    __shared__ unsigned long long block_first;
    const unsigned long long n = totals[0];
    if (n > 0xffffffffull) return;  // record keys hold 32 bits of work index; the host reports it
    const uint32_t wbits = work_bits(n);
    const unsigned long long stride = (unsigned long long)gridDim.x * blockDim.x;
    // The records' places in the buffer come from one atomic per workgroup and
    // trip: the counter is one address, which takes some 90 million atomics a
    // second, and with one per wave it was the kernel's bound. 128^3 x 6 levels,
    // 21 260 triangles: 54 us.
    for (unsigned long long base = (unsigned long long)blockIdx.x * 256u; base < n; base += stride) {
        const unsigned long long wi = base + threadIdx.x;
        Record out[6];
        int faces[6];
        int ic[3] = {0, 0, 0};
        int nout = 0, slot = 0;
        // one item: its records in `out`, `nout` of them
        auto raster = [&]() {
            const WorkItem it = work_item(E, totals, ntris, S.n, wi);
            slot = it.slot;
            if (!it.valid) return;
            const VoxParams P = S.P[it.slot];
            const float box_lo[3] = {S.box_lo[it.slot][0], S.box_lo[it.slot][1], S.box_lo[it.slot][2]};
            const float box_hi[3] = {S.box_hi[it.slot][0], S.box_hi[it.slot][1], S.box_hi[it.slot][2]};
            const uint32_t t = it.t;
            float p[9];
#pragma unroll
            for (int k = 0; k < 9; ++k) p[k] = pos[9u * t + k];
            TriSetup s;
            if (!tri_setup(p, P.voxel_size, P.samples, P.lo, P.hi, s)) return;
            float fp[3];
            double lam[3];
            if (!tri_sample(p, s, P.voxel_size, P.samples, it.sample, fp, lam)) return;
            if (fp[0] < box_lo[0] || fp[1] < box_lo[1] || fp[2] < box_lo[2] || fp[0] > box_hi[0] || fp[1] > box_hi[1] ||
                fp[2] > box_hi[2])
                return;
            const vct_gltf_material& m = T.mats[T.mat[t]];
            float uv[2] = {0.0f, 0.0f};
            if (T.tex) {
                // msaaInjectRadiance.frag:73-74: occlusion-texture discard
                interp_uv(T.uv + 6u * t, lam, uv);
                if (occluded(T, m, uv)) return;
            }
            image_coords(P, fp, ic);
            if (m.emissive_factor[0] > 0.0f || m.emissive_factor[1] > 0.0f || m.emissive_factor[2] > 0.0f) {
                // msaaInjectRadiance.frag:76-86; the emissive texture adds to the factor
                float em[3] = {m.emissive_factor[0], m.emissive_factor[1], m.emissive_factor[2]};
                if (has_texture(T, m.emissive_texture)) {
                    const f4 te = sample_texture(T.tex[m.emissive_texture], uv);
                    em[0] = em[0] + te.x;
                    em[1] = em[1] + te.y;
                    em[2] = em[2] + te.z;
                }
                Record e = {fminf(fmaxf(em[0], 0.0f), 1.0f), fminf(fmaxf(em[1], 0.0f), 1.0f),
                            fminf(fmaxf(em[2], 0.0f), 1.0f)};
                for (int f = 0; f < 6; ++f) {
                    out[f] = e;
                    faces[f] = f;
                }
                nout = 6;
            } else {
                // msaaInjectRadiance.frag:131-153
                const float* n0 = nrm + 9u * t;
                float ni[3];
                for (int k = 0; k < 3; ++k)
                    ni[k] = (float)(lam[0] * (double)n0[k] + lam[1] * (double)n0[3 + k] + lam[2] * (double)n0[6 + k]);
                const float len = sqrtf(ni[0] * ni[0] + ni[1] * ni[1] + ni[2] * ni[2]);
                const float nn[3] = {ni[0] / len, ni[1] / len, ni[2] / len};
                float ndl = nn[0] * L.dir[0] + nn[1] * L.dir[1] + nn[2] * L.dir[2];
                ndl = fminf(fmaxf(ndl, 0.001f), 1.0f);
                const float vis = visibility(L, fp, P.quirks);
                float lc[3];
                for (int k = 0; k < 3; ++k) lc[k] = ndl * vis * L.color[k] * L.intensity;
                if (lc[0] == 0.0f && lc[1] == 0.0f && lc[2] == 0.0f) return;
                // msaaInjectRadiance.frag:131-136: the base-colour texture scales the factor
                float col[4] = {m.base_color_factor[0], m.base_color_factor[1], m.base_color_factor[2],
                                m.base_color_factor[3]};
                if (has_texture(T, m.base_color_texture)) {
                    const f4 tb = sample_texture(T.tex[m.base_color_texture], uv);
                    col[0] = col[0] * tb.x;
                    col[1] = col[1] * tb.y;
                    col[2] = col[2] * tb.z;
                    col[3] = col[3] * tb.w;
                }
                float rad[3];
                for (int k = 0; k < 3; ++k) rad[k] = fminf(fmaxf(lc[k] * col[k] * col[3], 0.0f), 1.0f);
                const int face[3] = {(-nn[0] > 0.0f) ? 0 : 1, (-nn[1] > 0.0f) ? 2 : 3, (-nn[2] > 0.0f) ? 4 : 5};
                for (int k = 0; k < 3; ++k) {
                    const float w = fabsf(nn[k]);
                    out[k] = {rad[0] * w, rad[1] * w, rad[2] * w};
                    faces[k] = face[k];
                }
                nout = 3;
            }
        };
        if (wi < n) raster();  // n is a multiple of 64: whole waves
        slot = __builtin_amdgcn_readfirstlane(slot);
        const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
        uint32_t upto = (uint32_t)nout;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t u = __shfl_up(upto, off, 64);
            if (lane >= (uint32_t)off) upto += u;
        }
        __syncthreads();  // the previous trip's reads of the shared words are done
        if (lane == 63u) wave_records[wave] = upto;
        __syncthreads();
        if (threadIdx.x == 0) {
            const uint32_t all = wave_records[0] + wave_records[1] + wave_records[2] + wave_records[3];
            block_first = all ? atomicAdd(&totals[kTotRec], (unsigned long long)all) : 0ull;
        }
        __syncthreads();
        if (nout) {
            unsigned long long first = block_first + upto - (uint32_t)nout;
            for (uint32_t w = 0; w < wave; ++w) first += wave_records[w];
            const unsigned long long index = work_index(totals, slot, wi);
            const int D = S.P[slot].D, level = S.P[slot].clip_level;
#pragma unroll
            for (int j = 0; j < 6; ++j) {
                const unsigned long long r = first + (unsigned long long)j;
                if (j >= nout || r >= cap) break;  // capacity is checked on the host from the counter
                const size_t addr = vol_index(D, level, faces[j], ic[0], ic[1], ic[2]);
                keys[r] = ((unsigned long long)addr << wbits) | index;
                idx[r] = (uint32_t)r;
                vals[r] = out[j];
            }
        }
    }
}

// The state of a texel while its records are applied: the RGBA8 running
// average's channels and count as floats (rgba8_avg without the packing
// between records), or the FP32 sums and count of the half-float mean.
template <bool kHalf>
struct Applied {
    float x, y, z, w;

    __device__ __forceinline__ void add(float vx, float vy, float vz)
    {
#pragma clang fp contract(off)
        if (kHalf) {
            x = x + vx;
            y = y + vy;
            z = z + vz;
            w = w + 1.0f;
            return;
        }
        vx = vx * 255.0f;
        vy = vy * 255.0f;
        vz = vz * 255.0f;
        if (x == 0.0f && y == 0.0f && z == 0.0f && w == 0.0f) {
            x = byte(vx);
            y = byte(vy);
            z = byte(vz);
            w = 1.0f;
            return;
        }
        // the three quotients by the new count (1 to 256) from its correctly
        // rounded reciprocal and one residual correction each (Markstein's
        // theorem), which rounds as the division does and keeps it off the
        // chain from record to record (the reciprocal depends on the count only)
        const float d = w + 1.0f, r = 1.0f / d;
        x = average(x * w + vx, d, r);
        y = average(y * w + vy, d, r);
        z = average(z * w + vz, d, r);
        w = d == 256.0f ? 0.0f : d;  // the count is stored in a byte
    }

private:
    __device__ static __forceinline__ float average(float sum, float d, float r)
    {
        const float q = sum * r;
        return byte(__builtin_fmaf(__builtin_fmaf(-d, q, sum), r, q));
    }

    // the byte pack_raw keeps of a channel
    __device__ static __forceinline__ float byte(float v) { return (float)((uint32_t)v & 0xffu); }
};

template <bool kHalf>
__device__ __forceinline__ Applied<kHalf> apply_begin(const void* vol, unsigned long long addr)
{
    if (kHalf) return {0.0f, 0.0f, 0.0f, 0.0f};
    const f4 t = unpack_raw(((const uint32_t*)vol)[addr]);
    return {t.x, t.y, t.z, t.w};
}

template <bool kHalf>
__device__ __forceinline__ void apply_end(void* vol, unsigned long long addr, const Applied<kHalf>& A,
                                          uint32_t keep_mask, size_t level_texels)
{
    if (kHalf) {
        const bool keep = (keep_mask >> (uint32_t)(addr / level_texels)) & 1u;
        const float a = keep ? unpack_half(((const uint2*)vol)[addr]).w : 1.0f;
        ((uint2*)vol)[addr] = pack_half(f4{A.x / A.w, A.y / A.w, A.z / A.w, a});
    } else {
        ((uint32_t*)vol)[addr] = pack_raw(f4{A.x, A.y, A.z, A.w});
    }
}

// The texel's records in fragment order, applied as the reference's running
// average (RGBA8) or the FP32 sum / count mean (RGBA16F): one lane per run
// head of the sorted records. Runs are a few records but where a region's
// clamp collects thousands in one texel, and a record is two dependent loads
// (its index, then its value): the wave takes its runs of more than kShortRun
// records one by one, 64 records loaded at a time, the next ones while these
// are applied. A frame whose runs are long (64^3 x 5 levels RGBA8, 4 samples,
// camera off the room's centre): 193 us with one lane and one record at a
// time, now 70; 128^3 x 6 levels RGBA16F: 93 and 29 us.
constexpr uint32_t kShortRun = 8;

template <bool kHalf>
__global__ __launch_bounds__(256) void k_apply(const unsigned long long* __restrict__ keys,
                                               const uint32_t* __restrict__ idx, const Record* __restrict__ vals,
                                               uint32_t n, void* __restrict__ vol, uint32_t keep_mask, uint32_t wbits,
                                               size_t level_texels)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x, lane = threadIdx.x & 63u;
    const unsigned long long addr = i < n ? keys[i] >> wbits : 0ull;
    const bool head = i < n && (i == 0u || (keys[i - 1] >> wbits) != addr);
    const bool is_long = head && (unsigned long long)i + kShortRun < n && (keys[i + kShortRun] >> wbits) == addr;
    if (head && !is_long) {
        bool in[kShortRun];
        Record v[kShortRun];
#pragma unroll
        for (uint32_t k = 0; k < kShortRun; ++k) {
            in[k] = (unsigned long long)i + k < n && (keys[i + k] >> wbits) == addr;
            if (in[k]) v[k] = vals[idx[i + k]];
        }
        Applied<kHalf> A = apply_begin<kHalf>(vol, addr);
#pragma unroll
        for (uint32_t k = 0; k < kShortRun; ++k)
            if (in[k]) A.add(v[k].r, v[k].g, v[k].b);
        apply_end<kHalf>(vol, addr, A, keep_mask, level_texels);
    }
    for (unsigned long long todo = __ballot(is_long); todo != 0ull; todo &= todo - 1ull) {
        const int leader = __ffsll((long long)todo) - 1;
        const uint32_t first = __builtin_amdgcn_readlane(i, leader);
        const unsigned long long run =
            (unsigned long long)__builtin_amdgcn_readlane((uint32_t)addr, leader) |
            ((unsigned long long)__builtin_amdgcn_readlane((uint32_t)(addr >> 32), leader) << 32);
        // the run's records [j, j + 64), one per lane; a run is contiguous
        auto load = [&](unsigned long long j, Record& v) -> uint32_t {
            const bool in = j + lane < n && (keys[j + lane] >> wbits) == run;
            v = {0.0f, 0.0f, 0.0f};
            if (in) v = vals[idx[j + lane]];
            return (uint32_t)__popcll(__ballot(in));
        };
        Applied<kHalf> A = apply_begin<kHalf>(vol, run);
        Record v;
        uint32_t m = load(first, v);
        for (unsigned long long j = first; m != 0u; j += 64) {
            Record next = {0.0f, 0.0f, 0.0f};
            const uint32_t mn = m == 64u ? load(j + 64, next) : 0u;
            for (uint32_t k = 0; k < m; ++k) {
                auto lane_of = [&](float f) {
                    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f), (int)k));
                };
                A.add(lane_of(v.r), lane_of(v.g), lane_of(v.b));
            }
            v = next;
            m = mn;
        }
        if ((int)lane == leader) apply_end<kHalf>(vol, run, A, keep_mask, level_texels);
    }
}

static vct_status make_params(vct_ctx* c, const vct_voxelization_desc* d, uint32_t level, VoxParams* P)
{
    if (!d) return fail(VCT_ERR_INVALID_ARGUMENT, "null desc");
    if (level >= (uint32_t)c->levels || d->clip_level != level)
        return fail(VCT_ERR_INVALID_ARGUMENT, "level mismatch (desc %u, call %u)", d->clip_level, level);
    if (d->clipmap_resolution != c->res) return fail(VCT_ERR_INVALID_ARGUMENT, "clipmap_resolution");
    if (!(d->voxel_size > 0.0f) || !(d->clip_max_extent > 0.0f))
        return fail(VCT_ERR_INVALID_ARGUMENT, "voxel_size / clip_max_extent must be positive");
    for (int k = 0; k < 3; ++k) {
        P->region_min[k] = d->region_min_corner[k];
        P->region_max[k] = d->region_max_corner[k];
        // integer region recovered from the corners written by Voxelizer::cmdVoxelize
        const float lo = std::rint((d->region_min_corner[k] + 1e-6f) / d->voxel_size);
        const float hi = std::rint((d->region_max_corner[k] - 1e-6f) / d->voxel_size);
        if (!(std::fabs(lo) < 1e8f) || !(std::fabs(hi) < 1e8f) || hi < lo)
            return fail(VCT_ERR_INVALID_ARGUMENT, "region corners");
        P->lo[k] = (int)lo - 1;
        P->hi[k] = (int)hi;
    }
    P->clip_max_extent = d->clip_max_extent;
    P->voxel_size = d->voxel_size;
    P->clip_level = (int)level;
    P->res = c->res;
    P->D = c->D;
    P->samples = (int)c->cfg.raster_samples;
    P->quirks = c->cfg.quirks;
    return VCT_OK;
}

// The level set of `count` descriptors (their clip levels distinct), with
// each level's depth-clip box for the injection.
static vct_status make_level_set(vct_ctx* c, const vct_voxelization_desc* descs, uint32_t count, LevelSet* S)
{
    if (!descs || count == 0 || count > (uint32_t)kMaxLevels)
        return fail(VCT_ERR_INVALID_ARGUMENT, "1 to %d voxelization descriptors are required", kMaxLevels);
    std::memset(S, 0, sizeof(*S));
    uint32_t seen = 0;
    for (uint32_t i = 0; i < count; ++i) {
        const uint32_t level = descs[i].clip_level;
        if (level < 32u && (seen >> level) & 1u)
            return fail(VCT_ERR_INVALID_ARGUMENT, "clip level %u appears twice", level);
        VCT_TRY(make_params(c, &descs[i], level, &S->P[i]));
        seen |= 1u << level;
        for (int k = 0; k < 3; ++k) {
            S->box_lo[i][k] = (float)S->P[i].lo[k] * S->P[i].voxel_size;
            S->box_hi[i][k] = (float)(S->P[i].hi[k] + 1) * S->P[i].voxel_size;
        }
    }
    S->n = (int)count;
    return VCT_OK;
}

// The expansion of the (level, triangle) pairs and the totals.
static vct_status expand(vct_ctx* c, hipStream_t s, const TriSoup& soup, const LevelSet& S, Expansion* E)
{
    const uint32_t nblocks = (soup.count + kExpandBlock - 1u) / kExpandBlock;
    const size_t n = (size_t)nblocks * (size_t)S.n;
    if ((size_t)soup.count * (size_t)S.n > 0x7fffffffull)
        return fail(VCT_ERR_CAPACITY, "%zu triangle-level pairs exceed 2^31", (size_t)soup.count * (size_t)S.n);
    VCT_TRY(ensure(c->counts, 8u * (n ? n : 1) * kExpandBlock));
    VCT_TRY(ensure(c->offsets, 8u * (n ? n : 1)));
    VCT_TRY(ensure(c->totals, 8u * kTotWords));
    if (n)
        hipLaunchKernelGGL(k_count, dim3(nblocks, (unsigned)S.n), dim3(kExpandBlock), 0, s, soup.pos, soup.count, S,
                           (unsigned long long*)c->counts.ptr, (unsigned long long*)c->offsets.ptr);
    hipLaunchKernelGGL(k_total, dim3(1), dim3(1024), 0, s, (unsigned long long*)c->offsets.ptr, nblocks, S.n,
                       (unsigned long long*)c->totals.ptr);
    VCT_HIP(hipGetLastError());
    *E = {(const unsigned long long*)c->counts.ptr, (const unsigned long long*)c->offsets.ptr};
    return VCT_OK;
}

static vct_status voxelize_levels(vct_ctx* c, hipStream_t s, const vct_mesh* mesh, const vct_voxelization_desc* descs,
                                  uint32_t count)
{
    if (!c) return fail(VCT_ERR_INVALID_ARGUMENT, "null context");
    LevelSet S;
    VCT_TRY(make_level_set(c, descs, count, &S));
    TriSoup soup;
    VCT_TRY(run_vertex_stage(c, s, mesh, &soup, TextureUse::kSample, false));
    if (!soup.count) return VCT_OK;
    Expansion E;
    VCT_TRY(expand(c, s, soup, S, &E));
    // grid-stride over a device-side total: no host synchronisation
    const TexInputs T{soup.uv, soup.mat, mesh->materials, soup.tex, soup.tex_count};
    hipLaunchKernelGGL(k_raster_opacity, dim3(8192), dim3(256), 0, s, soup.pos, E, soup.count,
                       (const unsigned long long*)c->totals.ptr, S, T, (uint32_t*)c->opacity.ptr);
    VCT_HIP(hipGetLastError());
    return VCT_OK;
}

static vct_status inject_levels(vct_ctx* c, hipStream_t s, const vct_mesh* mesh, const vct_shadow_map* shadow,
                                const vct_directional_light_desc* light,
                                const vct_directional_light_shadow_desc* light_shadow,
                                const vct_voxelization_desc* descs, uint32_t count)
{
    if (!c) return fail(VCT_ERR_INVALID_ARGUMENT, "null context");
    if (!shadow || !shadow->depth || !shadow->width || !shadow->height || !light || !light_shadow)
        return fail(VCT_ERR_INVALID_ARGUMENT, "light, light_shadow and shadow map are required");
    LevelSet S;
    VCT_TRY(make_level_set(c, descs, count, &S));
    radiance_written(c);
    // after vct_begin_radiance_level the texels already carry the opacity alpha
    for (int i = 0; i < S.n; ++i) {
        const int level = S.P[i].clip_level;
        if (c->keep_alpha[level]) S.keep_mask |= 1u << level;
        c->keep_alpha[level] = false;
    }
    TriSoup soup;
    VCT_TRY(run_vertex_stage(c, s, mesh, &soup));
    if (!soup.count) return VCT_OK;
    Expansion E;
    VCT_TRY(expand(c, s, soup, S, &E));

    LightParams L;
    {
        // normalize(-uDirectionalLight.direction) with IEEE sqrt/div
        float nd[3] = {-light->direction[0], -light->direction[1], -light->direction[2]};
        float len = std::sqrt(nd[0] * nd[0] + nd[1] * nd[1] + nd[2] * nd[2]);
        for (int k = 0; k < 3; ++k) L.dir[k] = nd[k] / len;
        for (int k = 0; k < 3; ++k) L.color[k] = light->color[k];
        L.intensity = light->intensity;
        for (int k = 0; k < 16; ++k) {
            L.view[k] = light_shadow->view[k];
            L.proj[k] = light_shadow->proj[k];
        }
        L.z_near = light_shadow->z_near;
        L.z_far = light_shadow->z_far;
        L.depth = shadow->depth;
        L.width = (int)shadow->width;
        L.height = (int)shadow->height;
    }
    // The raster writes into a grow-only record buffer and counts every record
    // (those past the capacity are counted, not stored). One host read-back
    // of the count sizes the sort; a count above the capacity grows the
    // buffer and runs the raster again, which happens while the capacity
    // warms up. Record keys carry the work index, so the sorted order does
    // not depend on which run stored them.
    if (!c->pinned_word) VCT_HIP(hipHostMalloc(&c->pinned_word, kPinnedWordBytes, hipHostMallocDefault));
    volatile unsigned long long* landed = (volatile unsigned long long*)c->pinned_word;
    unsigned long long tot[2] = {0, 0};
    const TexInputs T{soup.uv, soup.mat, mesh->materials, soup.tex, soup.tex_count};
    for (int attempt = 0;; ++attempt) {
        const uint32_t cap = c->inject_cap;
        hipLaunchKernelGGL(k_raster_inject, dim3(8192), dim3(256), 0, s, soup.pos, soup.nrm, T, E, soup.count,
                           (unsigned long long*)c->totals.ptr,
                           S, L, (unsigned long long*)c->rec_key[0].ptr, (uint32_t*)c->rec_idx[0].ptr,
                           (Record*)c->rec_val.ptr, cap);
        VCT_HIP(hipGetLastError());
        VCT_HIP(hipMemcpyAsync((void*)landed, c->totals.ptr, 8u * kTotWords, hipMemcpyDeviceToHost, s));
        VCT_HIP(hipStreamSynchronize(s));
        tot[0] = landed[0];
        tot[1] = landed[kTotRec];
        if (tot[0] > 0xffffffffull) return fail(VCT_ERR_CAPACITY, "raster work %llu exceeds 2^32", tot[0]);
        if (tot[1] <= cap) break;
        if (tot[1] > 0xfffffff0ull || attempt > 0)
            return fail(VCT_ERR_CAPACITY, "injection records overflow (%llu > %u)", tot[1], cap);
        const unsigned long long want = tot[1] + tot[1] / 4 + 1024;
        const uint32_t grown = want > 0xfffffff0ull ? 0xfffffff0u : (uint32_t)want;
        for (int b = 0; b < 2; ++b) {
            VCT_TRY(ensure(c->rec_key[b], 8u * (size_t)grown));
            VCT_TRY(ensure(c->rec_idx[b], 4u * (size_t)grown));
        }
        VCT_TRY(ensure(c->rec_val, sizeof(Record) * (size_t)grown));
        c->inject_cap = grown;
        hipLaunchKernelGGL(k_reset_records, dim3(1), dim3(1), 0, s, (unsigned long long*)c->totals.ptr);
        VCT_HIP(hipGetLastError());
    }
    const uint32_t nrec = (uint32_t)tot[1];
    if (!nrec) return VCT_OK;
    // key bits: the texel index in the volume above the work index
    const uint32_t wbits = work_bits(tot[0]);
    const size_t level_texels = (size_t)kFaces * (size_t)c->D * (size_t)c->D * (size_t)c->D;
    const size_t volume_texels = level_texels * (size_t)c->levels;
    int end_bit = (int)wbits;
    while (end_bit < 64 && ((volume_texels - 1) >> (end_bit - (int)wbits)) != 0) ++end_bit;
    size_t tmp = 0;
    VCT_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp, (unsigned long long*)c->rec_key[0].ptr,
                                               (unsigned long long*)c->rec_key[1].ptr, (uint32_t*)c->rec_idx[0].ptr,
                                               (uint32_t*)c->rec_idx[1].ptr, (int)nrec, 0, end_bit, s));
    VCT_TRY(ensure(c->sort_tmp, tmp));
    VCT_HIP(hipcub::DeviceRadixSort::SortPairs(c->sort_tmp.ptr, tmp, (unsigned long long*)c->rec_key[0].ptr,
                                               (unsigned long long*)c->rec_key[1].ptr, (uint32_t*)c->rec_idx[0].ptr,
                                               (uint32_t*)c->rec_idx[1].ptr, (int)nrec, 0, end_bit, s));
    const bool half = c->cfg.radiance_format == VCT_FORMAT_RGBA16F;
    if (half)
        hipLaunchKernelGGL(k_apply<true>, dim3((nrec + 255) / 256), dim3(256), 0, s,
                           (const unsigned long long*)c->rec_key[1].ptr, (const uint32_t*)c->rec_idx[1].ptr,
                           (const Record*)c->rec_val.ptr, nrec, c->radiance.ptr, S.keep_mask, wbits, level_texels);
    else
        hipLaunchKernelGGL(k_apply<false>, dim3((nrec + 255) / 256), dim3(256), 0, s,
                           (const unsigned long long*)c->rec_key[1].ptr, (const uint32_t*)c->rec_idx[1].ptr,
                           (const Record*)c->rec_val.ptr, nrec, c->radiance.ptr, 0u, wbits, level_texels);
    VCT_HIP(hipGetLastError());
    return VCT_OK;
}

}  // namespace vct

using namespace vct;

extern "C" {

vct_status vct_voxelize_opacity(vct_ctx* c, vct_stream stream, const vct_mesh* mesh, const vct_voxelization_desc* d,
                                uint32_t level)
{
    if (d && d->clip_level != level)
        return fail(VCT_ERR_INVALID_ARGUMENT, "level mismatch (desc %u, call %u)", d->clip_level, level);
    return voxelize_levels(c, (hipStream_t)stream, mesh, d, 1);
}

vct_status vct_voxelize_opacity_levels(vct_ctx* c, vct_stream stream, const vct_mesh* mesh,
                                       const vct_voxelization_desc* descs, uint32_t count)
{
    return voxelize_levels(c, (hipStream_t)stream, mesh, descs, count);
}

vct_status vct_inject_radiance(vct_ctx* c, vct_stream stream, const vct_mesh* mesh, const vct_shadow_map* shadow,
                               const vct_directional_light_desc* light,
                               const vct_directional_light_shadow_desc* light_shadow,
                               const vct_voxelization_desc* d, uint32_t level)
{
    if (d && d->clip_level != level)
        return fail(VCT_ERR_INVALID_ARGUMENT, "level mismatch (desc %u, call %u)", d->clip_level, level);
    return inject_levels(c, (hipStream_t)stream, mesh, shadow, light, light_shadow, d, 1);
}

vct_status vct_inject_radiance_levels(vct_ctx* c, vct_stream stream, const vct_mesh* mesh,
                                      const vct_shadow_map* shadow, const vct_directional_light_desc* light,
                                      const vct_directional_light_shadow_desc* light_shadow,
                                      const vct_voxelization_desc* descs, uint32_t count)
{
    return inject_levels(c, (hipStream_t)stream, mesh, shadow, light, light_shadow, descs, count);
}

}  // extern "C"
