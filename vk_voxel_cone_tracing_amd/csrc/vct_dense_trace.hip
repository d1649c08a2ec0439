// vct_dense_trace.hip - cone tracing over the dense mip pyramid (gfx950).
//
// Per pixel: the reference's 16 (or 32) diffuse cones (voxelConeTracing.frag
// :166-203) marched through the dense pyramid; output RGBA32F =
// (indirect diffuse x albedo x intensity, ambient occlusion). Level 0 has one
// face, so its sample is one trilinear fetch scaled by the weight sum; levels
// >= 1 blend the three direction-selected faces. Every face block has a zero
// border, so only positions more than one texel outside the grid need a test.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "vct_dense.hpp"
#include "vct_dense_march.hpp"

namespace vct {
namespace dense {

// The images of one launch: one view, or the views of a tape call (one image
// size, each with its own camera, G-buffer, output and tape).
constexpr int kTraceViews = 16;
struct TraceViews {
    float vp_inv[kTraceViews][16];
    const uint32_t* diffuse[kTraceViews];
    const uint16_t* normal[kTraceViews];
    const float* depth[kTraceViews];
    float4* out[kTraceViews];
    float4* tape[kTraceViews];
    uint8_t* counts[kTraceViews];
};

// One pixel per lane, one view of 8x8-pixel waves in 16x16 tiles per
// workgroup of blockIdx.y, kWaves waves to an 8x8 tile. With one wave (four
// 8x8 tiles to a workgroup) a lane marches every cone of its pixel. With
// more, the waves share the tile's cones, leaving each cone's result in LDS
// ([cone][lane], dynamic), and the first adds them in cone order, so the
// images are the same bit for bit. kTape (RGBA32F grids): every accumulated
// sample of every cone is also written, in the (wave, cone) slot layout of
// TapeLayout, with each lane's step count per cone.
// Register budget of four waves per SIMD: a 512x512 view with one wave per
// tile is 1024 workgroups, one round of four waves per SIMD, so a five-wave
// budget buys no occupancy and only makes the scheduler keep fewer texel
// loads in flight (64 views of 512x512: 28.8 -> 22.6 ms).
template <bool kF32, int kWaves, bool kTape>
__global__ __launch_bounds__(kWaves == 1 ? 256 : 64 * kWaves) __attribute__((amdgpu_waves_per_eu(4, 4))) void
k_dense_trace(const void* __restrict__ data, Pyramid P, March M, TraceViews VW, int width, int height,
              unsigned long long* __restrict__ samples, uint32_t cap)
{
    extern __shared__ f4 cones[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned tiles_x = ((unsigned)width + 15u) / 16u, v = blockIdx.y;
    const unsigned block = xcd_remap(blockIdx.x, gridDim.x);
    const unsigned tile = kWaves == 1 ? block : block >> 2, sub = kWaves == 1 ? (unsigned)wave : block & 3u;
    const int px = (int)(tile % tiles_x) * 16 + (int)(sub & 1u) * 8 + (lane & 7);
    const int py = (int)(tile / tiles_x) * 16 + (int)(sub >> 1) * 8 + (lane >> 3);
    const bool in_image = px < width && py < height;
    const size_t idx = (size_t)py * (size_t)width + (size_t)px;
    const float depth = in_image ? VW.depth[v][idx] : 1.0f;
    const bool surface = depth != 1.0f;
    const int first = kWaves == 1 ? 0 : wave;
    const size_t slot0 = ((size_t)tile * 4u + (size_t)sub) * (size_t)M.ncones;
    float4* const col = kTape ? VW.tape[v] + slot0 * cap * 64u + lane : nullptr;
    uint8_t* const counts = kTape ? VW.counts[v] + slot0 * 64u + lane : nullptr;
    uint32_t steps = 0;
    float start[3], normal[3], albedo[3];
    f4 ind = {0.0f, 0.0f, 0.0f, 1.0f};
    auto add_cone = [&](const f4& c, float ct) {
        ind.x += c.x * ct;
        ind.y += c.y * ct;
        ind.z += c.z * ct;
        ind.w += c.w * ct;
    };
    if (surface) {
#pragma unroll
        for (int k = 0; k < 16; ++k) M.vp_inv[k] = VW.vp_inv[v][k];
        pixel_setup(P, M, px, py, width, height, depth, VW.normal[v] + 4 * idx, VW.diffuse[v][idx], start, normal, albedo);
    }
    for (int i = first; i < M.ncones; i += kWaves) {
        uint32_t n = 0;
        if (surface) {
            const float* d = cone_dir(M, i);
            const float ct = normal[0] * d[0] + normal[1] * d[1] + normal[2] * d[2];
            if (ct >= 0.0f) {
                TapeSlot t{kTape ? col + (size_t)i * cap * 64u : nullptr, cap, 0u};
                const f4 c = march<kF32, false>(data, P, M, start, d, steps, kTape ? &t : nullptr);
                n = t.count > cap ? kTapeOverflow : t.count;
                if (kWaves == 1) add_cone(c, ct);
                else cones[i * 64 + lane] = c;
            }
        }
        if (kTape) counts[i * 64] = (uint8_t)n;
    }
    if (kWaves > 1) __syncthreads();
    if ((kWaves == 1 || wave == 0) && in_image) {
        float4 o = make_float4(0.0f, 0.0f, 0.0f, 1.0f);
        if (surface) {
            if (kWaves > 1)
                for (int i = 0; i < M.ncones; ++i) {
                    const float* d = cone_dir(M, i);
                    const float ct = normal[0] * d[0] + normal[1] * d[1] + normal[2] * d[2];
                    if (ct >= 0.0f) add_cone(cones[i * 64 + lane], ct);
                }
            const float inv = 1.0f / (float)M.ncones;
            o = make_float4(ind.x * inv * albedo[0] * M.diffuse_intensity, ind.y * inv * albedo[1] * M.diffuse_intensity,
                            ind.z * inv * albedo[2] * M.diffuse_intensity, ind.w * inv * M.ao_factor);
        }
        VW.out[v][idx] = o;
    }
    if (samples) {
        unsigned long long n = steps;
        for (int off = 32; off > 0; off >>= 1) n += __shfl_down(n, off, 64);
        if (lane == 0 && n) atomicAdd(samples, n);
    }
}

// 8x8 tiles (of all views) up to which sixteen and four waves share a tile: one
// workgroup of sixteen waves for each of the 256 CUs, and two rounds of four
// one-wave tiles per SIMD. One wave / four (sixteen at 200x160), whole plain
// VXAO frame at 128^3: 200x160 268 / 141 us, 320x180 265 / 165, 480x270 287 /
// 223, 640x360 355 / 302, 960x540 (8160 tiles) 545 / 521, 1280x720 797 / 818.
constexpr uint64_t kWideTiles = 256, kSplitTiles = 8192;

template <bool kF32, int kWaves, bool kTape>
static void launch_waves(hipStream_t s, const void* data, const Pyramid& P, const March& M, const TraceViews& VW,
                         uint32_t views, uint32_t width, uint32_t height, unsigned long long* samples, uint32_t cap)
{
    const unsigned tiles = ((width + 15) / 16) * ((height + 15) / 16);
    const size_t lds = kWaves == 1 ? 0 : (size_t)M.ncones * 64u * sizeof(f4);
    hipLaunchKernelGGL((k_dense_trace<kF32, kWaves, kTape>), dim3(kWaves == 1 ? tiles : 4u * tiles, views),
                       dim3(kWaves == 1 ? 256 : 64 * kWaves), lds, s, data, P, M, VW, (int)width, (int)height, samples,
                       cap);
}

template <bool kF32, bool kTape>
static void launch_trace(hipStream_t s, const void* data, const Pyramid& P, const March& M, const TraceViews& VW,
                         uint32_t views, uint32_t width, uint32_t height, unsigned long long* samples, uint32_t cap)
{
    const uint64_t tiles = 4ull * views * ((width + 15) / 16) * ((height + 15) / 16);
    if (tiles <= kWideTiles) launch_waves<kF32, 16, kTape>(s, data, P, M, VW, views, width, height, samples, cap);
    else if (tiles <= kSplitTiles) launch_waves<kF32, 4, kTape>(s, data, P, M, VW, views, width, height, samples, cap);
    else launch_waves<kF32, 1, kTape>(s, data, P, M, VW, views, width, height, samples, cap);
}

}  // namespace dense
}  // namespace vct

using namespace vct;

// `views` views of one image size, kTraceViews to a launch; tapes may be null.
static vct_status trace_views(vct_dense* g, hipStream_t s, uint32_t views, const vct_gbuffer* gbs,
                              const vct_camera_ubo* cams, const vct_dense_trace_desc* d, float* const* outs,
                              void* const* tapes, size_t tape_bytes, unsigned long long* samples)
{
    if (!g || !d) return fail(VCT_ERR_INVALID_ARGUMENT, "null argument");
    if (!views) return VCT_OK;  // the arrays of no views may be null (an empty vector's data())
    if (!gbs || !cams || !outs) return fail(VCT_ERR_INVALID_ARGUMENT, "null argument");
    const uint32_t W = gbs[0].width, H = gbs[0].height;
    for (uint32_t v = 0; v < views; ++v) {
        if (!outs[v] || (tapes && !tapes[v])) return fail(VCT_ERR_INVALID_ARGUMENT, "null argument");
        if (!gbs[v].diffuse || !gbs[v].normal || !gbs[v].depth || !gbs[v].width || !gbs[v].height)
            return fail(VCT_ERR_INVALID_ARGUMENT, "G-buffer needs diffuse, normal and depth");
        if (gbs[v].width != W || gbs[v].height != H)
            return fail(VCT_ERR_INVALID_ARGUMENT, "views differ in image size");
    }
    if (tapes && g->texel_bytes != 16) return fail(VCT_ERR_UNSUPPORTED, "the adjoint tape needs an RGBA32F grid");
    dense::Pyramid P;
    dense::March M;
    VCT_TRY(dense::make_params(g, &cams[0], d, &P, &M));
    dense::TapeLayout T{};
    if (tapes) {
        T = dense::tape_layout(P, M, W, H, dense::kSweepHeaderBytes);
        if (T.cap > (uint32_t)dense::kAdjMaxSteps)
            return fail(VCT_ERR_UNSUPPORTED, "the march takes more than %d steps", dense::kAdjMaxSteps - 2);
        if (tape_bytes < T.bytes)
            return fail(VCT_ERR_INVALID_ARGUMENT, "the tape holds %zu bytes; this view's takes %zu", tape_bytes, T.bytes);
        if ((T.sample_bytes / sizeof(float4)) >> 32) return fail(VCT_ERR_UNSUPPORTED, "tape above 2^32 samples");
        for (uint32_t v = 0; v < views; ++v)
            if ((uintptr_t)tapes[v] % 16u) return fail(VCT_ERR_INVALID_ARGUMENT, "the tape must be 16-byte aligned");
    }
    for (uint32_t v0 = 0; v0 < views; v0 += dense::kTraceViews) {
        const uint32_t n = std::min<uint32_t>(views - v0, dense::kTraceViews);
        dense::TraceViews VW{};
        for (uint32_t k = 0; k < n; ++k) {
            const uint32_t v = v0 + k;
            for (int e = 0; e < 16; ++e) VW.vp_inv[k][e] = cams[v].view_proj_inv[e];
            VW.diffuse[k] = gbs[v].diffuse;
            VW.normal[k] = gbs[v].normal;
            VW.depth[k] = gbs[v].depth;
            VW.out[k] = (float4*)outs[v];
            if (tapes) {
                VW.tape[k] = (float4*)tapes[v];
                VW.counts[k] = (uint8_t*)tapes[v] + T.sample_bytes;
            }
        }
        if (tapes) dense::launch_trace<true, true>(s, g->data.ptr, P, M, VW, n, W, H, samples, T.cap);
        else if (g->texel_bytes == 16) dense::launch_trace<true, false>(s, g->data.ptr, P, M, VW, n, W, H, samples, 0u);
        else dense::launch_trace<false, false>(s, g->data.ptr, P, M, VW, n, W, H, samples, 0u);
    }
    VCT_HIP(hipGetLastError());
    return VCT_OK;
}

extern "C" vct_status vct_dense_trace(vct_dense* g, vct_stream stream, const vct_gbuffer* gb,
                                      const vct_camera_ubo* cam, const vct_dense_trace_desc* d, float* out,
                                      unsigned long long* samples_out)
{
    return trace_views(g, (hipStream_t)stream, 1, gb, cam, d, &out, nullptr, 0, samples_out);
}

extern "C" vct_status vct_dense_trace_views(vct_dense* g, vct_stream stream, uint32_t views, const vct_gbuffer* gbs,
                                            const vct_camera_ubo* cams, const vct_dense_trace_desc* d,
                                            float* const* outs, void* const* tapes, size_t tape_bytes)
{
    return trace_views(g, (hipStream_t)stream, views, gbs, cams, d, outs, tapes, tape_bytes, nullptr);
}

extern "C" vct_status vct_dense_tape_bytes(vct_dense* g, const vct_gbuffer* gb, const vct_camera_ubo* cam,
                                           const vct_dense_trace_desc* d, size_t* bytes)
{
    if (!g || !gb || !cam || !d || !bytes) return fail(VCT_ERR_INVALID_ARGUMENT, "null argument");
    if (!gb->width || !gb->height) return fail(VCT_ERR_INVALID_ARGUMENT, "empty G-buffer");
    dense::Pyramid P;
    dense::March M;
    VCT_TRY(dense::make_params(g, cam, d, &P, &M));
    const dense::TapeLayout T = dense::tape_layout(P, M, gb->width, gb->height, dense::kSweepHeaderBytes);
    if (T.cap > (uint32_t)dense::kAdjMaxSteps)
        return fail(VCT_ERR_UNSUPPORTED, "the march takes more than %d steps", dense::kAdjMaxSteps - 2);
    *bytes = T.bytes;
    return VCT_OK;
}

extern "C" vct_status vct_dense_trace_tape(vct_dense* g, vct_stream stream, const vct_gbuffer* gb,
                                           const vct_camera_ubo* cam, const vct_dense_trace_desc* d, float* out,
                                           unsigned long long* samples_out, void* tape, size_t tape_bytes)
{
    if (!tape) return fail(VCT_ERR_INVALID_ARGUMENT, "null argument");
    return trace_views(g, (hipStream_t)stream, 1, gb, cam, d, &out, &tape, tape_bytes, samples_out);
}
