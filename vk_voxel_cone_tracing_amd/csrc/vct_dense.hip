// vct_dense.hip - the "plain" dense-grid method on gfx950: one res^3 grid
// voxelized from triangles, a 6-face anisotropic mip pyramid down to 1^3, and
// the cone march for ambient occlusion + indirect diffuse.
//
// This applies the reference's kernels (dominant-axis voxelization,
// radianceDownSample's front-to-back pairs, traceCone) to a single dense grid
// instead of a clipmap; the level rule is clamp(log2(diameter / voxelSize),
// 0, levels - 1). Storage per level m: level 0 keeps one face (all six faces
// are equal after voxelization), levels >= 1 keep six faces; every face block
// carries a one-texel zero border so the trilinear footprint never needs a
// bounds test inside the grid. Texels are RGBA8 or RGBA32F.
#include <hip/hip_runtime.h>

#include <cmath>
#include <new>

#include "vct_dense.hpp"
#include "vct_dense_mip.hpp"
#include "vct_expand.hpp"
#include "vct_internal.hpp"
#include "vct_raster.hpp"
#include "vct_texel.hpp"

static_assert(sizeof(vct_dense_desc) == 32, "vct_dense_desc layout");
static_assert(sizeof(vct_dense_trace_desc) == 32, "vct_dense_trace_desc layout");

namespace vct {

vct_status dense_alloc(vct_dense* g)
{
    size_t total = 0;
    for (int m = 0; m < g->nlevels; ++m) {
        g->offset[m] = total;
        const int n = g->res >> m;
        g->block[m] = (size_t)(n + 2) * (n + 2) * (n + 2);
        total += g->block[m] * (m == 0 ? 1u : 6u);
    }
    g->texels = total;
    return ensure(g->data, total * g->texel_bytes);
}

struct DenseRaster {
    float vs;
    int lo[3], hi[3];
    int samples;
    int res;
};

// A triangle in grid coordinates (written to tpos) and its item count, scanned
// within the workgroup's 256 triangles.
__global__ __launch_bounds__(kExpandBlock) void k_dense_count(const float* __restrict__ pos, uint32_t ntris, float mx,
                                                              float my, float mz, DenseRaster R,
                                                              float* __restrict__ tpos,
                                                              unsigned long long* __restrict__ in_block,
                                                              unsigned long long* __restrict__ block_sums)
{
#pragma clang fp contract(off)
    const uint32_t t = blockIdx.x * kExpandBlock + threadIdx.x;
    unsigned long long n = 0;
    if (t < ntris) {
        float p[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            p[k] = pos[9u * t + k] - (k % 3 == 0 ? mx : (k % 3 == 1 ? my : mz));
            tpos[9u * t + k] = p[k];
        }
        TriSetup s;
        if (tri_setup(p, R.vs, R.samples, R.lo, R.hi, s))
            n = (unsigned long long)s.nu * s.nv * (unsigned long long)R.samples;
    }
    const unsigned long long below = expand_block(n, &block_sums[blockIdx.x]);
    in_block[blockIdx.x * kExpandBlock + threadIdx.x] = below;
}

__global__ __launch_bounds__(1024) void k_dense_total(unsigned long long* __restrict__ blocks, uint32_t nblocks,
                                                      unsigned long long* __restrict__ total)
{
    const unsigned long long all = expand_scan(blocks, nblocks);
    if (threadIdx.x == 0) total[0] = all;
}

__global__ void k_fill_u32(uint32_t* __restrict__ p, size_t n, uint32_t v)
{
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Every covered sample proposes its triangle for its voxel; the smallest
// triangle index (the first fragment in rasterization order) wins.
__global__ __launch_bounds__(256) void k_dense_raster(const float* __restrict__ tpos, Expansion E, uint32_t ntris,
                                                      const unsigned long long* __restrict__ total, DenseRaster R,
                                                      uint32_t* __restrict__ winner)
{
#pragma clang fp contract(off)
    const unsigned long long n = total[0];
    const unsigned long long stride = (unsigned long long)gridDim.x * blockDim.x;
    // whole waves: the search takes all 64 lanes
    for (unsigned long long first = (unsigned long long)blockIdx.x * blockDim.x + (threadIdx.x & ~63u); first < n;
         first += stride) {
        const uint32_t t = wave_triangle(E, ntris, first, n - 1ull);
        const unsigned long long wi = first + (threadIdx.x & 63u);
        if (wi >= n) continue;
        float p[9];
        for (int k = 0; k < 9; ++k) p[k] = tpos[9u * t + k];
        TriSetup s;
        if (!tri_setup(p, R.vs, R.samples, R.lo, R.hi, s)) continue;
        float fp[3];
        double lam[3];
        if (!tri_sample(p, s, R.vs, R.samples, (uint32_t)(wi - E(t)), fp, lam)) continue;
        int ic[3];
        bool inside = true;
        for (int k = 0; k < 3; ++k) {
            const float f = floorf(fp[k] / R.vs);
            if (!(f >= 0.0f) || f >= (float)R.res) inside = false;
            ic[k] = (int)f;
        }
        if (!inside) continue;
        atomicMin(&winner[((size_t)ic[2] * R.res + ic[1]) * R.res + ic[0]], t);
    }
}

// The winners' colours into level 0; every winner is returned to empty for the
// next voxelization. A thread takes kPer consecutive voxels of a row (4 of a
// row of at least 4: one 16-byte read, and nearly all are empty). Bound by the
// read of the winners. 256^3: 51 us with one voxel a thread and divisions by
// the resolution, 32 us so; the fill of the winners before each voxelization
// (18 us) is gone.
template <bool kF32, int kPer>
__global__ __launch_bounds__(256) void k_dense_resolve(uint32_t* __restrict__ winner, const uint32_t* __restrict__ mat,
                                                       const vct_gltf_material* __restrict__ mats, int log2_res,
                                                       void* __restrict__ level0)
{
    const uint32_t v = (blockIdx.x * 256u + threadIdx.x) * kPer, res = 1u << log2_res;  // res <= 1024
    if (v >> (3 * log2_res)) return;
    uint32_t t[kPer];
    if (kPer == 4) {
        const uint4 q = *(const uint4*)(winner + v);
        if ((q.x & q.y & q.z & q.w) == 0xffffffffu) return;
        t[0] = q.x;
        t[1 % kPer] = q.y;
        t[2 % kPer] = q.z;
        t[3 % kPer] = q.w;
    } else {
        t[0] = winner[v];
    }
    const uint32_t x = v & (res - 1u), y = (v >> log2_res) & (res - 1u), z = v >> (2 * log2_res);
    const size_t D = (size_t)res + 2;
    const size_t i = ((size_t)(z + 1) * D + (size_t)(y + 1)) * D + (size_t)(x + 1);
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        if (t[k] == 0xffffffffu) continue;
        winner[v + k] = 0xffffffffu;
        const float* bc = mats[mat[t[k]]].base_color_factor;
        if (kF32) ((float4*)level0)[i + k] = make_float4(bc[0], bc[1], bc[2], 1.0f);
        else ((uint32_t*)level0)[i + k] = pack_unorm(f4{bc[0], bc[1], bc[2], 1.0f});
    }
}

// radianceDownSample.comp:95-139 over the whole grid. Level 1 (kFirst): one
// thread per destination texel, all six faces from one read of its children.
// The other levels: one thread per texel and face (blockIdx.z also counts the
// faces), so that no thread's loads wait for another face's stores. Bound by
// HBM from 64^3 up. 256^3 grid, RGBA8: level 1 166 us with the children read
// and divided by 255 once per face, now 28 (120 MB, 4.2 TB/s), level 2 24 -> 12
// us; RGBA32F: level 1 177 -> 98 us (470 MB, 4.8 TB/s), level 2 46 -> 37.
template <bool kF32, bool kFirst>
__global__ __launch_bounds__(256) void k_dense_mip(const void* __restrict__ src, void* __restrict__ dst, int n,
                                                   int zblocks)
{
    const int f = kFirst ? 0 : (int)blockIdx.z / zblocks;
    const int x = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const int y = (int)(blockIdx.y * blockDim.y + threadIdx.y);
    const int z = ((int)blockIdx.z - f * zblocks) * (int)blockDim.z + (int)threadIdx.z;
    if (x >= n || y >= n || z >= n) return;
    if (kFirst) dense_mip_first<kF32>(src, dst, n, x, y, z);
    else dense_mip_texel<kF32>(src, dst, n, x, y, z, f);
}

struct MipOffsets {
    unsigned long long at[11];
};

template <bool kF32>
__global__ __launch_bounds__(512) void k_dense_mip_tail(void* data, MipOffsets O, int res, int m, int nlevels)
{
    dense_mip_tail<kF32>(data, O.at, res, m, nlevels, (int)blockIdx.x);
}

template <bool kF32>
static void launch_mips(const vct_dense* g, hipStream_t s)
{
    char* data = (char*)g->data.ptr;
    for (int m = 1; m < g->nlevels; ++m) {
        const int n = g->res >> m;
        if (n <= tail_edge<kF32>()) {
            MipOffsets O;
            for (int l = 0; l < g->nlevels; ++l) O.at[l] = g->offset[l];
            hipLaunchKernelGGL(k_dense_mip_tail<kF32>, dim3(kFaces), dim3(512), 0, s, (void*)data, O, g->res, m,
                               g->nlevels);
            return;
        }
        const dim3 block(n < 64 ? n : 64, 2, 2);
        const unsigned zblocks = (unsigned)(n + 1) / 2;
        const dim3 grid((n + block.x - 1) / block.x, (n + 1) / 2, zblocks * (m == 1 ? 1u : (unsigned)kFaces));
        const void* src = data + g->offset[m - 1] * g->texel_bytes;
        void* dst = data + g->offset[m] * g->texel_bytes;
        if (m == 1) hipLaunchKernelGGL((k_dense_mip<kF32, true>), grid, block, 0, s, src, dst, n, (int)zblocks);
        else hipLaunchKernelGGL((k_dense_mip<kF32, false>), grid, block, 0, s, src, dst, n, (int)zblocks);
    }
}

}  // namespace vct

using namespace vct;

extern "C" {

vct_status vct_dense_create(vct_dense** out, const vct_dense_desc* d)
{
    if (!out || !d) return fail(VCT_ERR_INVALID_ARGUMENT, "null argument");
    *out = nullptr;
    const uint32_t r = d->resolution;
    if (r < 2 || r > 1024 || (r & (r - 1))) return fail(VCT_ERR_INVALID_ARGUMENT, "resolution must be a power of two in [2, 1024]");
    if (d->format != VCT_FORMAT_RGBA8 && d->format != VCT_FORMAT_RGBA32F)
        return fail(VCT_ERR_INVALID_ARGUMENT, "format must be RGBA8 or RGBA32F");
    if (!(d->extent > 0.0f)) return fail(VCT_ERR_INVALID_ARGUMENT, "extent must be positive");
    if (d->raster_samples != 1 && d->raster_samples != 4) return fail(VCT_ERR_INVALID_ARGUMENT, "raster_samples");
    vct_dense* g = new (std::nothrow) vct_dense();
    if (!g) return fail(VCT_ERR_OUT_OF_MEMORY, "host allocation failed");
    g->desc = *d;
    g->res = (int)r;
    int n = 0;
    while ((1u << n) < r) ++n;
    g->nlevels = n + 1;
    g->texel_bytes = d->format == VCT_FORMAT_RGBA32F ? 16u : 4u;
    vct_config cfg{8, 0, VCT_FORMAT_RGBA8, 0, d->raster_samples, 0, 1.0f, 0};
    vct_status s = vct_create(&g->scratch, &cfg);
    if (s == VCT_OK) s = dense_alloc(g);
    if (s == VCT_OK) {
        hipError_t e = hipMemset(g->data.ptr, 0, g->texels * g->texel_bytes);
        if (e == hipSuccess) e = hipDeviceSynchronize();
        if (e != hipSuccess) s = fail(VCT_ERR_HIP, "clear failed: %s", hipGetErrorString(e));
    }
    if (s != VCT_OK) {
        vct_dense_destroy(g);
        return s;
    }
    *out = g;
    return VCT_OK;
}

vct_status vct_dense_destroy(vct_dense* g)
{
    if (!g) return VCT_OK;
    (void)hipDeviceSynchronize();
    release(g->data);
    release(g->winner);
    release(g->bwd_rec);
    release(g->bwd_hdr);
    release(g->bwd_start);
    release(g->bwd_ctr);
    if (g->scratch) vct_destroy(g->scratch);
    delete g;
    return VCT_OK;
}

vct_status vct_dense_clear(vct_dense* g, vct_stream stream)
{
    if (!g) return fail(VCT_ERR_INVALID_ARGUMENT, "null grid");
    VCT_HIP(hipMemsetAsync(g->data.ptr, 0, g->texels * g->texel_bytes, (hipStream_t)stream));
    return VCT_OK;
}

vct_status vct_dense_level(vct_dense* g, uint32_t level, void** ptr, size_t* bytes, uint32_t* faces)
{
    if (!g || !ptr) return fail(VCT_ERR_INVALID_ARGUMENT, "null argument");
    if (level >= (uint32_t)g->nlevels) return fail(VCT_ERR_INVALID_ARGUMENT, "level out of range");
    *ptr = (char*)g->data.ptr + g->offset[level] * g->texel_bytes;
    if (bytes) *bytes = g->block[level] * (level == 0 ? 1u : 6u) * g->texel_bytes;
    if (faces) *faces = level == 0 ? 1u : 6u;
    return VCT_OK;
}

// Voxelizes a mesh into level 0: opacity 1 and the base colour of the first
// triangle (in draw order) that covers the voxel.
vct_status vct_dense_voxelize(vct_dense* g, vct_stream stream, const vct_mesh* mesh)
{
    if (!g) return fail(VCT_ERR_INVALID_ARGUMENT, "null grid");
    hipStream_t s = (hipStream_t)stream;
    vct_ctx* c = g->scratch;
    TriSoup soup;
    VCT_TRY(run_vertex_stage(c, s, mesh, &soup, TextureUse::kRefuse, false));
    if (!soup.count) return VCT_OK;
    VCT_TRY(ensure(c->rec_val, 36u * (size_t)soup.count));
    float* tpos = (float*)c->rec_val.ptr;
    DenseRaster R;
    R.vs = g->desc.extent / (float)g->res;
    for (int k = 0; k < 3; ++k) {
        R.lo[k] = 0;
        R.hi[k] = g->res - 1;
    }
    R.samples = (int)g->desc.raster_samples;
    R.res = g->res;
    const uint32_t nblocks = (soup.count + kExpandBlock - 1u) / kExpandBlock;
    VCT_TRY(ensure(c->counts, 8u * (size_t)nblocks * kExpandBlock));
    VCT_TRY(ensure(c->offsets, 8u * (size_t)nblocks));
    VCT_TRY(ensure(c->totals, 64));
    const size_t nv = (size_t)g->res * g->res * g->res;
    VCT_TRY(ensure(g->winner, 4u * nv));
    // Every voxelization leaves the winners empty for the next; one that fails
    // on the way leaves that to the next. A fill that is only recorded into a
    // graph runs with the graph, so the calls after it fill again.
    const bool fill = !g->winners_empty;
    bool recorded = false;
    g->winners_empty = false;
    if (fill) {
        hipStreamCaptureStatus capture;
        VCT_HIP(hipStreamIsCapturing(s, &capture));
        recorded = capture != hipStreamCaptureStatusNone;
        hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)((nv + 255) / 256)), dim3(256), 0, s, (uint32_t*)g->winner.ptr,
                           nv, 0xffffffffu);
    }
    const Expansion E{(const unsigned long long*)c->counts.ptr, (const unsigned long long*)c->offsets.ptr};
    auto* total = (unsigned long long*)c->totals.ptr;
    hipLaunchKernelGGL(k_dense_count, dim3(nblocks), dim3(kExpandBlock), 0, s, soup.pos, soup.count,
                       g->desc.grid_min[0], g->desc.grid_min[1], g->desc.grid_min[2], R, tpos,
                       (unsigned long long*)c->counts.ptr, (unsigned long long*)c->offsets.ptr);
    hipLaunchKernelGGL(k_dense_total, dim3(1), dim3(1024), 0, s, (unsigned long long*)c->offsets.ptr, nblocks, total);
    hipLaunchKernelGGL(k_dense_raster, dim3(8192), dim3(256), 0, s, (const float*)tpos, E, soup.count,
                       (const unsigned long long*)total, R, (uint32_t*)g->winner.ptr);
    int log2_res = 0;
    while ((1 << log2_res) < g->res) ++log2_res;
    auto resolve = [&](auto kernel, size_t per) {
        const size_t threads = (nv + per - 1) / per;
        hipLaunchKernelGGL(kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s,
                           (uint32_t*)g->winner.ptr, soup.mat, mesh->materials, log2_res, g->data.ptr);
    };
    if (g->texel_bytes == 16) g->res >= 4 ? resolve(k_dense_resolve<true, 4>, 4) : resolve(k_dense_resolve<true, 1>, 1);
    else g->res >= 4 ? resolve(k_dense_resolve<false, 4>, 4) : resolve(k_dense_resolve<false, 1>, 1);
    VCT_HIP(hipGetLastError());
    g->winners_empty = !recorded;
    return VCT_OK;
}

// Builds levels 1..log2(res) from level 0 (DownSampler applied per level).
vct_status vct_dense_mipmap(vct_dense* g, vct_stream stream)
{
    if (!g) return fail(VCT_ERR_INVALID_ARGUMENT, "null grid");
    hipStream_t s = (hipStream_t)stream;
    if (g->texel_bytes == 16) launch_mips<true>(g, s);
    else launch_mips<false>(g, s);
    VCT_HIP(hipGetLastError());
    return VCT_OK;
}

vct_status vct_dense_read_level(vct_dense* g, vct_stream stream, uint32_t level, void* dst, size_t bytes)
{
    void* p;
    size_t b;
    VCT_TRY(vct_dense_level(g, level, &p, &b, nullptr));
    if (!dst || bytes != b) return fail(VCT_ERR_INVALID_ARGUMENT, "buffer is %zu bytes, level is %zu", bytes, b);
    VCT_HIP(hipMemcpyAsync(dst, p, b, hipMemcpyDeviceToHost, (hipStream_t)stream));
    VCT_HIP(hipStreamSynchronize((hipStream_t)stream));
    return VCT_OK;
}

vct_status vct_dense_write_level(vct_dense* g, vct_stream stream, uint32_t level, const void* src, size_t bytes)
{
    void* p;
    size_t b;
    VCT_TRY(vct_dense_level(g, level, &p, &b, nullptr));
    if (!src || bytes != b) return fail(VCT_ERR_INVALID_ARGUMENT, "buffer is %zu bytes, level is %zu", bytes, b);
    VCT_HIP(hipMemcpyAsync(p, src, b, hipMemcpyHostToDevice, (hipStream_t)stream));
    VCT_HIP(hipStreamSynchronize((hipStream_t)stream));
    return VCT_OK;
}

}  // extern "C"
