// vct_svo.hip - sparse voxel octree path for gfx950: fragment-list
// voxelization (K9), the per-level node init/flag/alloc build (K10-K13), leaf
// and mipmap colour writes (K14/K15) and octree cone tracing (K16).
//
// Determinism. The reference hands out fragment-list slots and child blocks
// with atomicAdd, so its layout depends on invocation order. Here:
//  * every covered raster sample gets its slot from an exclusive scan over the
//    (triangle, cell, sample) work items, i.e. rasterization order;
//  * child blocks are handed to the flagged nodes of a level in pool-index
//    order, which is the reference's outcome when invocations run in index
//    order: with the fragments sorted by leaf path, a node's place follows
//    from its rank among the distinct path prefixes of its depth;
//  * the order-dependent leaf running average is applied per leaf in
//    fragment order (the sort by path is stable).
// The node pool is therefore a pure function of the fragment list.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <cmath>
#include <vector>

#include "vct_expand.hpp"
#include "vct_internal.hpp"
#include "vct_raster.hpp"
#include "vct_shadow.hpp"
#include "vct_texel.hpp"
#include "vct_textures.hpp"

namespace vct {

struct SvoRaster {
    float vs;  // 2 / R: one raster cell per voxel of the normalised [-1, 1] box
    int lo[3], hi[3];
    int samples;
    int res;
    uint32_t quirks;
};

// The triangle in the normalised box (written to npos) and its raster samples,
// scanned within the workgroup's 256 triangles.
__global__ __launch_bounds__(kExpandBlock) void k_svo_count(const float* __restrict__ pos, uint32_t ntris, float cx,
                                                            float cy, float cz, float ev, SvoRaster R,
                                                            float* __restrict__ npos,
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
            p[k] = (pos[9u * t + k] - (k % 3 == 0 ? cx : (k % 3 == 1 ? cy : cz))) / ev;  // voxelizer.vert:42-47
            npos[9u * t + k] = p[k];
        }
        TriSetup s;
        if (tri_setup(p, R.vs, R.samples, R.lo, R.hi, s))
            n = (unsigned long long)s.nu * s.nv * (unsigned long long)R.samples;
    }
    const unsigned long long below = expand_block(n, &block_sums[blockIdx.x]);
    in_block[blockIdx.x * kExpandBlock + threadIdx.x] = below;
}

// Exclusive prefix of n sums in place, and their total.
__global__ __launch_bounds__(1024) void k_svo_scan(unsigned long long* __restrict__ sums, uint32_t n,
                                                   unsigned long long* __restrict__ total)
{
    const unsigned long long all = expand_scan(sums, n);
    if (threadIdx.x == 0) total[0] = all;
}

constexpr uint32_t kCoverItems = 1024;  // work items per workgroup of k_svo_cover

// The covered samples: each is one fragment invocation and consumes one
// fragment-list slot (voxelizer.frag:55). A workgroup leaves its own, as
// (triangle, local work item) in order, at the start of its 1024 places in
// staged, and their number in counts. The fragment pass reads triangle and item
// back instead of searching for them. 1M triangles at 2^9 per axis: 235 us with
// a search of 20 steps per lane and a flag per work item, 190 us so; the scan of
// the flags and the compaction of their slots 230 us, of the workgroups 30 us.
__global__ __launch_bounds__(256) void k_svo_cover(const float* __restrict__ npos, Expansion E, uint32_t ntris,
                                                   uint32_t nwork, SvoRaster R, TexInputs T,
                                                   uint2* __restrict__ staged,
                                                   unsigned long long* __restrict__ counts)
{
    constexpr uint32_t kWaveItems = kCoverItems / 4u;
    __shared__ uint2 s_entry[4][kWaveItems];
    __shared__ uint32_t s_count[4];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const unsigned long long block0 = (unsigned long long)blockIdx.x * kCoverItems;
    uint32_t mine = 0;
#pragma unroll 1
    for (uint32_t c = 0; c < kWaveItems / 64u; ++c) {
        const unsigned long long first = block0 + wave * kWaveItems + c * 64u;
        if (first >= nwork) break;
        const uint32_t t = wave_triangle(E, ntris, first, (unsigned long long)nwork - 1ull);
        bool covered = false;
        uint32_t local = 0;
        if (first + lane < nwork) {
            float p[9];
            for (int k = 0; k < 9; ++k) p[k] = npos[9u * t + k];
            TriSetup s;
            if (tri_setup(p, R.vs, R.samples, R.lo, R.hi, s)) {
                float fp[3];
                double lam[3];
                local = (uint32_t)(first + lane - E(t));
                covered = tri_sample(p, s, R.vs, R.samples, local, fp, lam);
                if (covered && T.tex) {
                    // voxelizer.frag:52-53: occlusion-texture discard, before the slot
                    float uv[2];
                    interp_uv(T.uv + 6u * t, lam, uv);
                    if (occluded(T, T.mats[T.mat[t]], uv)) covered = false;
                }
            }
        }
        const unsigned long long m = __ballot(covered);
        if (covered) s_entry[wave][mine + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = make_uint2(t, local);
        mine += (uint32_t)__popcll(m);
    }
    if (lane == 0u) s_count[wave] = mine;
    __syncthreads();
    uint32_t below = 0;
    for (uint32_t w = 0; w < wave; ++w) below += s_count[w];
    for (uint32_t i = lane; i < mine; i += 64u) staged[block0 + below + i] = s_entry[wave][i];
    if (threadIdx.x == 255u) counts[blockIdx.x] = (unsigned long long)(below + mine);
}

// Every fragment's triangle and work item: the workgroups' lists end to end.
__global__ __launch_bounds__(256) void k_svo_compact(const uint2* __restrict__ staged,
                                                     const unsigned long long* __restrict__ offsets, uint32_t nblocks,
                                                     uint32_t nfrag, uint2* __restrict__ list)
{
    const uint32_t at = (uint32_t)offsets[blockIdx.x];
    const uint32_t n = (blockIdx.x + 1u < nblocks ? (uint32_t)offsets[blockIdx.x + 1u] : nfrag) - at;
    for (uint32_t i = threadIdx.x; i < n; i += 256u) list[at + i] = staged[(size_t)blockIdx.x * kCoverItems + i];
}

// voxelizer.frag:48-100, one thread per fragment (so every lane of a wave
// has a fragment to light), in fragment order.
__global__ __launch_bounds__(256) void k_svo_write(const float* __restrict__ npos, const float* __restrict__ nrm,
                                                   TexInputs T, uint32_t nfrag, SvoRaster R, LightParams L,
                                                   const uint2* __restrict__ list, uint2* __restrict__ frags)
{
#pragma clang fp contract(off)
    const uint32_t cur = blockIdx.x * blockDim.x + threadIdx.x;
    if (cur >= nfrag) return;
    const uint2 item = list[cur];
    const uint32_t t = item.x;
    float p[9];
    for (int k = 0; k < 9; ++k) p[k] = npos[9u * t + k];
    TriSetup s;
    if (!tri_setup(p, R.vs, R.samples, R.lo, R.hi, s)) return;
    float fp[3];
    double lam[3];
    if (!tri_sample(p, s, R.vs, R.samples, item.y, fp, lam)) return;
    float q[3];
    for (int k = 0; k < 3; ++k) q[k] = (fp[k] + 1.0f) * 0.5f;  // biasAndScale (voxelizer.geom:27-30)
    const vct_gltf_material& m = T.mats[T.mat[t]];
    float uv[2] = {0.0f, 0.0f};
    if (T.tex) interp_uv(T.uv + 6u * t, lam, uv);
    float rad[4] = {1.0f, 1.0f, 1.0f, 1.0f};
    if (m.emissive_factor[0] > 0.0f || m.emissive_factor[1] > 0.0f || m.emissive_factor[2] > 0.0f) {
        // voxelizer.frag:60-69; the emissive texture adds to the factor
        float em[3] = {m.emissive_factor[0], m.emissive_factor[1], m.emissive_factor[2]};
        if (has_texture(T, m.emissive_texture)) {
            const f4 te = sample_texture(T.tex[m.emissive_texture], uv);
            em[0] = em[0] + te.x;
            em[1] = em[1] + te.y;
            em[2] = em[2] + te.z;
        }
        for (int k = 0; k < 3; ++k) rad[k] = fminf(fmaxf(em[k], 0.0f), 1.0f);
    } else {
        // voxelizer.frag:72-77: texture x factor (black without a texture
        // under VCT_QUIRK_SVO_UNTEXTURED_BLACK)
        float color[4] = {0.0f, 0.0f, 0.0f, 1.0f};
        if (!(R.quirks & VCT_QUIRK_SVO_UNTEXTURED_BLACK) || m.base_color_texture > -1)
            for (int k = 0; k < 4; ++k) color[k] = m.base_color_factor[k];
        if (has_texture(T, m.base_color_texture)) {
            const f4 tb = sample_texture(T.tex[m.base_color_texture], uv);
            color[0] = tb.x * color[0];
            color[1] = tb.y * color[1];
            color[2] = tb.z * color[2];
            color[3] = tb.w * color[3];
        }
        const float* n0 = nrm + 9u * t;
        float ni[3];
        for (int k = 0; k < 3; ++k)
            ni[k] = (float)(lam[0] * (double)n0[k] + lam[1] * (double)n0[3 + k] + lam[2] * (double)n0[6 + k]);
        const float len = sqrtf(ni[0] * ni[0] + ni[1] * ni[1] + ni[2] * ni[2]);
        const float nn[3] = {ni[0] / len, ni[1] / len, ni[2] / len};
        float ndl = nn[0] * L.dir[0] + nn[1] * L.dir[1] + nn[2] * L.dir[2];
        ndl = fminf(fmaxf(ndl, 0.001f), 1.0f);
        // calcVisibility at fs_in.position, the normalised [0,1] position (voxelizer.frag:86)
        const float vis = visibility(L, q, R.quirks);
        float lc[3];
        for (int k = 0; k < 3; ++k) lc[k] = ndl * vis * L.color[k] * L.intensity;
        if (lc[0] == 0.0f && lc[1] == 0.0f && lc[2] == 0.0f) return;  // discard: the slot stays zero
        for (int k = 0; k < 3; ++k) rad[k] = fminf(fmaxf(lc[k] * color[k] * color[3], 0.0f), 1.0f);
        rad[3] = 1.0f;
    }
    uint32_t vp[3];
    for (int k = 0; k < 3; ++k) {
        const float f = q[k] * (float)R.res;
        uint32_t u = f > 0.0f ? (uint32_t)f : 0u;
        vp[k] = u > (uint32_t)R.res ? (uint32_t)R.res : u;
    }
    const f4 v255 = {rad[0] * 255.0f, rad[1] * 255.0f, rad[2] * 255.0f, rad[3] * 255.0f};
    frags[cur] = make_uint2(vp[0] | (vp[1] << 12u) | ((vp[2] & 0xffu) << 24u),
                            ((vp[2] >> 8u) << 28u) | (pack_raw(v255) & 0x0fffffffu));
}

__global__ void k_fill_u2(uint2* __restrict__ p, uint32_t n, uint2 v)
{
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

__device__ __forceinline__ void frag_pos(uint2 f, bool half, uint32_t p[3])
{
    p[0] = f.x & 0xfffu;
    p[1] = (f.x >> 12u) & 0xfffu;
    p[2] = ((f.x >> 24u) & 0xffu) | ((f.y >> 20u) & 0xf00u);
    if (half) {
        p[0] >>= 1;
        p[1] >>= 1;
        p[2] >>= 1;
    }
}

// The descent shared by octreeNodeFlag/LeafWrite/MipmapWrite.
__device__ __forceinline__ uint32_t walk(const uint2* __restrict__ pool, uint32_t p[3], uint32_t res, uint32_t stop,
                                         uint32_t& res_out)
{
    uint32_t idx = 0, cur = 0;
    do {
        res >>= 1;
        const uint32_t cx = p[0] >= res, cy = p[1] >= res, cz = p[2] >= res;
        idx = cur + (cz | (cx << 1) | (cy << 2));
        cur = pool[idx].x & 0x7fffffffu;
        p[0] -= cx * res;
        p[1] -= cy * res;
        p[2] -= cz * res;
    } while (cur != 0u && res > stop);
    res_out = res;
    return idx;
}

// The tree is built from the fragments sorted by their leaf's path: the child
// slots from the root down (z | x << 1 | y << 2 per depth, as in walk()), most
// significant first. octreeNodeAlloc hands out child blocks in pool order, and
// the nodes of a depth lie in the order of their parents' blocks, so by
// induction the pool order of a depth's nodes is the order of their paths. The
// nodes that some fragment reaches at depth e are the distinct prefixes of
// e + 1 slots; one's rank among them, and the number G_e of such nodes above
// depth e, give its child block (G_e + rank + 1) << 3, and its parent's block
// and its last slot give its index. One sort, one counting pass and one
// writing pass build every depth, with one read-back of the sizes, where a
// flag pass over all fragments (with atomics), an allocation (count, scan,
// assign) and a read-back per depth were needed. 2^9 per axis, 1M triangles:
// nine flag passes 880 us, nine allocations 190 us, leaf keys and averages 156
// us and a sort of 50-bit keys 290 us, now keys 16 us, a sort of 27-bit keys
// with their colours 245 us, counts 19 us and nodes with averages 82 us. Bound
// by the sort's passes over memory.

// A coordinate of 2^L takes walk()'s path for 2^L - 1.
template <typename Key>
__global__ __launch_bounds__(256) void k_svo_keys(const uint2* __restrict__ frags, uint32_t nfrag, uint32_t L,
                                                  bool half, Key* __restrict__ keys, uint32_t* __restrict__ colors)
{
    const uint32_t f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= nfrag) return;
    const uint2 v = frags[f];
    uint32_t p[3];
    frag_pos(v, half, p);
    const uint32_t top = (1u << L) - 1u;
    auto spread = [](uint32_t c) -> Key {  // bit b to bit 3b (the Morton code's steps)
        uint32_t r = c & 1023u;
        r = (r | (r << 16)) & 0x030000ffu;
        r = (r | (r << 8)) & 0x0300f00fu;
        r = (r | (r << 4)) & 0x030c30c3u;
        r = (r | (r << 2)) & 0x09249249u;
        Key k = r;
        if (sizeof(Key) == 8) k |= (Key)(c >> 10) << (sizeof(Key) == 8 ? 30 : 0);
        return k;
    };
    keys[f] = spread(min(p[2], top)) | (spread(min(p[0], top)) << 1) | (spread(min(p[1], top)) << 2);
    colors[f] = v.y & 0x0fffffffu;
}

constexpr uint32_t kSvoMaxDepth = 11;  // octree levels
constexpr uint32_t kNodeKeys = 1024;   // sorted fragments per workgroup, 256 per wave in four chunks

// The first depth at which sorted fragment i reaches another node than
// fragment i - 1 (L where both reach one leaf; L also past the last fragment).
template <typename Key>
__device__ __forceinline__ uint32_t first_new_depth(const Key* __restrict__ keys, uint32_t i, uint32_t n, uint32_t L,
                                                    Key& key)
{
    key = 0;
    if (i >= n) return L;
    key = keys[i];
    if (i == 0) return 0u;
    const unsigned long long d = (unsigned long long)(key ^ keys[i - 1]);
    return d ? L - 1u - (63u - (uint32_t)__clzll((long long)d)) / 3u : L;
}

// New nodes per depth of every workgroup's fragments: counts[depth][workgroup].
template <typename Key>
__global__ __launch_bounds__(256) void k_svo_node_count(const Key* __restrict__ keys, uint32_t n, uint32_t L,
                                                        unsigned long long* __restrict__ counts)
{
    __shared__ uint32_t s_count[4][kSvoMaxDepth];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t first = blockIdx.x * kNodeKeys + wave * (kNodeKeys / 4u);
    uint32_t mine[kSvoMaxDepth] = {};
#pragma unroll
    for (uint32_t c = 0; c < kNodeKeys / 256u; ++c) {
        Key key;
        const uint32_t f = first_new_depth(keys, first + c * 64u + lane, n, L, key);
#pragma unroll
        for (uint32_t e = 0; e < kSvoMaxDepth; ++e)
            if (e < L) mine[e] += (uint32_t)__popcll(__ballot(f <= e));
    }
    if (lane == 0u)
        for (uint32_t e = 0; e < L; ++e) s_count[wave][e] = mine[e];
    __syncthreads();
    if (threadIdx.x < L)
        counts[(size_t)threadIdx.x * gridDim.x + blockIdx.x] =
            (unsigned long long)s_count[0][threadIdx.x] + s_count[1][threadIdx.x] + s_count[2][threadIdx.x] +
            s_count[3][threadIdx.x];
}

// One workgroup per depth: the prefix of its counts over the workgroups, and
// the depth's number of nodes.
__global__ __launch_bounds__(1024) void k_svo_node_scan(unsigned long long* __restrict__ counts, uint32_t nblocks,
                                                        unsigned long long* __restrict__ totals)
{
    const unsigned long long all = expand_scan(counts + (size_t)blockIdx.x * nblocks, nblocks);
    if (threadIdx.x == 0) totals[blockIdx.x] = all;
}

// Every node some fragment reaches, written by the first of its fragments (the
// pool is zero before), and each leaf's running average over its fragments in
// fragment order (octreeNodeLeafWrite.comp; the sort is stable).
template <typename Key>
__global__ __launch_bounds__(256) void k_svo_nodes(const Key* __restrict__ keys, const uint32_t* __restrict__ colors,
                                                   uint32_t n, uint32_t L,
                                                   const unsigned long long* __restrict__ counts,
                                                   const unsigned long long* __restrict__ totals,
                                                   uint2* __restrict__ pool)
{
    __shared__ uint32_t s_count[4][kSvoMaxDepth];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t first = blockIdx.x * kNodeKeys + wave * (kNodeKeys / 4u);
    constexpr uint32_t kChunks = kNodeKeys / 256u;
    uint32_t f[kChunks], rank[kSvoMaxDepth] = {};
    Key key[kChunks];
#pragma unroll
    for (uint32_t c = 0; c < kChunks; ++c) {
        f[c] = first_new_depth(keys, first + c * 64u + lane, n, L, key[c]);
#pragma unroll
        for (uint32_t e = 0; e < kSvoMaxDepth; ++e)
            if (e < L) rank[e] += (uint32_t)__popcll(__ballot(f[c] <= e));
    }
    if (lane == 0u)
        for (uint32_t e = 0; e < L; ++e) s_count[wave][e] = rank[e];
    __syncthreads();
    // nodes of each depth begun before this wave's first fragment
#pragma unroll
    for (uint32_t e = 0; e < kSvoMaxDepth; ++e)
        if (e < L) {
            rank[e] = (uint32_t)counts[(size_t)e * gridDim.x + blockIdx.x];
            for (uint32_t w = 0; w < wave; ++w) rank[e] += s_count[w][e];
        }
    const unsigned long long upto = ~0ull >> (63u - lane);  // this lane and those below
#pragma unroll
    for (uint32_t c = 0; c < kChunks; ++c) {
        uint32_t block = 0;   // the child block that depth e's node lies in
        uint32_t above = 0;   // G_e
#pragma unroll
        for (uint32_t e = 0; e < kSvoMaxDepth; ++e) {
            if (e >= L) continue;
            const unsigned long long m = __ballot(f[c] <= e);
            const uint32_t child = (above + rank[e] + (uint32_t)__popcll(m & upto)) << 3;
            const uint32_t idx = block + ((uint32_t)(key[c] >> (3u * (L - 1u - e))) & 7u);
            if (f[c] <= e) {
                uint2 node = make_uint2(child | 0x80000000u, 0u);
                if (e == L - 1u) {
                    node.x = 0x80000000u;
                    for (uint32_t i = first + c * 64u + lane; i < n && keys[i] == key[c]; ++i)
                        node.y = rgba8_avg(node.y, unpack_raw(colors[i]));
                }
                pool[idx] = node;
            }
            block = child;
            above += (uint32_t)totals[e];
            rank[e] += (uint32_t)__popcll(m);
        }
    }
}

// octreeNodeMipmapWrite.comp evaluated per node: every flagged node of the
// depth range gets the truncating average of its eight children. The
// reference reaches exactly these nodes (the ancestors of fragments) once per
// fragment and writes the same value each time.
__global__ __launch_bounds__(256) void k_svo_mip(uint2* __restrict__ pool, uint32_t begin, uint32_t num)
{
#pragma clang fp contract(off)
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= num) return;
    const uint2 node = pool[begin + i];
    if (!(node.x & 0x80000000u)) return;
    const uint32_t child = node.x & 0x7fffffffu;
    if (child == 0u) return;
    float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (uint32_t j = 0; j < 8; ++j) {
        const f4 v = unpack_raw(pool[child + j].y);
        s[0] = s[0] + v.x / 8.0f;
        s[1] = s[1] + v.y / 8.0f;
        s[2] = s[2] + v.z / 8.0f;
        s[3] = s[3] + v.w / 8.0f;
    }
    pool[begin + i].y = pack_raw(f4{s[0], s[1], s[2], s[3]});
}

// The walk of every cell of 2^kSvoTopBits voxels, from the root: the state a
// sample's walk has on entering the cell, or where it ends above it.
__global__ __launch_bounds__(256) void k_svo_top(const uint2* __restrict__ pool, uint32_t L, uint32_t bits,
                                                 uint2* __restrict__ top)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x, mask = (1u << bits) - 1u;
    if (i >= 1u << (3u * bits)) return;
    uint32_t p[3] = {(i & mask) << kSvoTopBits, ((i >> bits) & mask) << kSvoTopBits, (i >> (2u * bits)) << kSvoTopBits};
    uint32_t r;
    const uint32_t idx = walk(pool, p, 1u << L, 1u << kSvoTopBits, r);
    const uint2 node = pool[idx];
    top[i] = make_uint2(r == 1u << kSvoTopBits ? node.x & 0x7fffffffu : 0u, node.y);
}

static LightParams make_light(const vct_shadow_map* shadow, const vct_directional_light_desc* light,
                              const vct_directional_light_shadow_desc* ls)
{
    LightParams L{};
    float nd[3] = {-light->direction[0], -light->direction[1], -light->direction[2]};
    float len = std::sqrt(nd[0] * nd[0] + nd[1] * nd[1] + nd[2] * nd[2]);
    for (int k = 0; k < 3; ++k) {
        L.dir[k] = nd[k] / len;
        L.color[k] = light->color[k];
    }
    L.intensity = light->intensity;
    for (int k = 0; k < 16; ++k) {
        L.view[k] = ls->view[k];
        L.proj[k] = ls->proj[k];
    }
    L.z_near = ls->z_near;
    L.z_far = ls->z_far;
    L.depth = shadow->depth;
    L.width = (int)shadow->width;
    L.height = (int)shadow->height;
    return L;
}

static unsigned blocks_for(uint64_t n, unsigned threads = 256)
{
    return (unsigned)((n + threads - 1) / threads);
}

// The fragments sorted by path (keys in rec_key[1], colours in rec_idx[1]) and
// the new nodes per depth: totals[depth], scanned per workgroup in counts.
template <typename Key>
static vct_status svo_sort(vct_ctx* c, hipStream_t s, const uint2* frags, uint32_t nfrag, uint32_t L, bool half)
{
    const uint32_t nblocks = blocks_for(nfrag, kNodeKeys);
    for (int b = 0; b < 2; ++b) {
        VCT_TRY(ensure(c->rec_key[b], sizeof(Key) * (size_t)nfrag));
        VCT_TRY(ensure(c->rec_idx[b], 4u * (size_t)nfrag));
    }
    VCT_TRY(ensure(c->counts, 8u * (size_t)L * nblocks));
    VCT_TRY(ensure(c->totals, 8u * kSvoMaxDepth));
    Key* k0 = (Key*)c->rec_key[0].ptr;
    Key* k1 = (Key*)c->rec_key[1].ptr;
    uint32_t* v0 = (uint32_t*)c->rec_idx[0].ptr;
    uint32_t* v1 = (uint32_t*)c->rec_idx[1].ptr;
    hipLaunchKernelGGL(k_svo_keys<Key>, dim3(blocks_for(nfrag)), dim3(256), 0, s, frags, nfrag, L, half, k0, v0);
    size_t tmp = 0;
    VCT_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp, k0, k1, v0, v1, (int)nfrag, 0, (int)(3u * L), s));
    VCT_TRY(ensure(c->sort_tmp, tmp));
    VCT_HIP(hipcub::DeviceRadixSort::SortPairs(c->sort_tmp.ptr, tmp, k0, k1, v0, v1, (int)nfrag, 0, (int)(3u * L), s));
    hipLaunchKernelGGL(k_svo_node_count<Key>, dim3(nblocks), dim3(256), 0, s, (const Key*)k1, nfrag, L,
                       (unsigned long long*)c->counts.ptr);
    hipLaunchKernelGGL(k_svo_node_scan, dim3(L), dim3(1024), 0, s, (unsigned long long*)c->counts.ptr, nblocks,
                       (unsigned long long*)c->totals.ptr);
    VCT_HIP(hipGetLastError());
    return VCT_OK;
}

template <typename Key>
static void svo_nodes(vct_ctx* c, hipStream_t s, uint32_t nfrag, uint32_t L, uint2* pool)
{
    hipLaunchKernelGGL(k_svo_nodes<Key>, dim3(blocks_for(nfrag, kNodeKeys)), dim3(256), 0, s,
                       (const Key*)c->rec_key[1].ptr, (const uint32_t*)c->rec_idx[1].ptr, nfrag, L,
                       (const unsigned long long*)c->counts.ptr, (const unsigned long long*)c->totals.ptr, pool);
}

}  // namespace vct

using namespace vct;

extern "C" {

// SparseVoxelizer::preVoxelize + cmdVoxelize (SparseVoxelizer.cpp:248-326).
vct_status vct_svo_voxelize(vct_ctx* c, vct_stream stream, const vct_mesh* mesh, const vct_shadow_map* shadow,
                            const vct_directional_light_desc* light,
                            const vct_directional_light_shadow_desc* light_shadow, uint32_t octree_level,
                            uint32_t* nfrag_out)
{
    if (!c || !mesh || !shadow || !shadow->depth || !light || !light_shadow)
        return fail(VCT_ERR_INVALID_ARGUMENT, "null argument");
    if (octree_level < 1 || octree_level > 11)
        return fail(VCT_ERR_INVALID_ARGUMENT, "octree_level must be in [1, 11] (EngineConfig.h:20-21)");
    hipStream_t s = (hipStream_t)stream;
    TriSoup soup;
    VCT_TRY(run_vertex_stage(c, s, mesh, &soup));
    const uint32_t R = 1u << octree_level;
    c->svo.level = octree_level;
    c->svo.built = false;
    c->svo.nfrag = 0;
    if (nfrag_out) *nfrag_out = 0;
    if (!soup.count) return VCT_OK;
    // voxelizer.vert:42-47 normalisation
    float ext[3], center[3];
    for (int k = 0; k < 3; ++k) {
        ext[k] = mesh->scene_bb_max[k] - mesh->scene_bb_min[k];
        center[k] = (mesh->scene_bb_min[k] + mesh->scene_bb_max[k]) * 0.5f;
    }
    const float ev = std::fmax(ext[0], std::fmax(ext[1], ext[2])) * 0.5f;
    if (!(ev > 0.0f)) return fail(VCT_ERR_INVALID_ARGUMENT, "empty scene bounding box");
    VCT_TRY(ensure(c->rec_val, 36u * (size_t)soup.count));
    float* npos = (float*)c->rec_val.ptr;
    SvoRaster Rr;
    Rr.vs = 2.0f / (float)R;
    for (int k = 0; k < 3; ++k) {
        Rr.lo[k] = -(int)(R / 2);
        Rr.hi[k] = (int)(R / 2) - 1;
    }
    Rr.samples = (int)c->cfg.raster_samples;
    Rr.res = (int)R;
    Rr.quirks = c->cfg.quirks;
    const uint32_t tri_blocks = blocks_for(soup.count, kExpandBlock);
    VCT_TRY(ensure(c->counts, 8u * (size_t)tri_blocks * kExpandBlock));
    VCT_TRY(ensure(c->offsets, 8u * (size_t)tri_blocks));
    VCT_TRY(ensure(c->totals, 64));
    const Expansion E{(const unsigned long long*)c->counts.ptr, (const unsigned long long*)c->offsets.ptr};
    hipLaunchKernelGGL(k_svo_count, dim3(tri_blocks), dim3(kExpandBlock), 0, s, soup.pos, soup.count, center[0],
                       center[1], center[2], ev, Rr, npos, (unsigned long long*)c->counts.ptr,
                       (unsigned long long*)c->offsets.ptr);
    hipLaunchKernelGGL(k_svo_scan, dim3(1), dim3(1024), 0, s, (unsigned long long*)c->offsets.ptr, tri_blocks,
                       (unsigned long long*)c->totals.ptr);
    if (!c->pinned_word) VCT_HIP(hipHostMalloc(&c->pinned_word, kPinnedWordBytes, hipHostMallocDefault));
    volatile unsigned long long* landed = (volatile unsigned long long*)c->pinned_word;
    VCT_HIP(hipMemcpyAsync((void*)landed, c->totals.ptr, 8, hipMemcpyDeviceToHost, s));
    VCT_HIP(hipStreamSynchronize(s));
    const unsigned long long nwork64 = landed[0];
    if (nwork64 >= 0xffffffffull) return fail(VCT_ERR_CAPACITY, "raster work %llu exceeds 2^32", nwork64);
    const uint32_t nwork = (uint32_t)nwork64;
    if (!nwork) return VCT_OK;
    const uint32_t cover_blocks = blocks_for(nwork, kCoverItems);
    VCT_TRY(ensure(c->rec_idx[0], 8u * (size_t)nwork));
    VCT_TRY(ensure(c->rec_idx[1], 8u * (size_t)cover_blocks));
    uint2* staged = (uint2*)c->rec_idx[0].ptr;
    auto* cover_counts = (unsigned long long*)c->rec_idx[1].ptr;
    const TexInputs T{soup.uv, soup.mat, mesh->materials, soup.tex, soup.tex_count};
    hipLaunchKernelGGL(k_svo_cover, dim3(cover_blocks), dim3(256), 0, s, (const float*)npos, E, soup.count, nwork, Rr, T,
                       staged, cover_counts);
    // the count pass's host read-back (SparseVoxelizer.cpp:279)
    hipLaunchKernelGGL(k_svo_scan, dim3(1), dim3(1024), 0, s, cover_counts, cover_blocks,
                       (unsigned long long*)c->totals.ptr);
    VCT_HIP(hipMemcpyAsync((void*)landed, c->totals.ptr, 8, hipMemcpyDeviceToHost, s));
    VCT_HIP(hipStreamSynchronize(s));
    const uint32_t nfrag = (uint32_t)landed[0];
    VCT_TRY(ensure(c->svo.frags, 8u * (size_t)(nfrag ? nfrag : 1)));
    if (nfrag) {
        hipLaunchKernelGGL(k_fill_u2, dim3(blocks_for(nfrag)), dim3(256), 0, s, (uint2*)c->svo.frags.ptr, nfrag,
                           make_uint2(0u, 0u));
        const LightParams L = make_light(shadow, light, light_shadow);
        VCT_TRY(ensure(c->rec_key[0], 8u * (size_t)nfrag));
        uint2* list = (uint2*)c->rec_key[0].ptr;
        hipLaunchKernelGGL(k_svo_compact, dim3(cover_blocks), dim3(256), 0, s, (const uint2*)staged,
                           (const unsigned long long*)cover_counts, cover_blocks, nfrag, list);
        hipLaunchKernelGGL(k_svo_write, dim3(blocks_for(nfrag)), dim3(256), 0, s, (const float*)npos, soup.nrm, T, nfrag,
                           Rr, L, (const uint2*)list, (uint2*)c->svo.frags.ptr);
        VCT_HIP(hipGetLastError());
    }
    c->svo.nfrag = nfrag;
    if (nfrag_out) *nfrag_out = nfrag;
    return VCT_OK;
}

// ---- 3^3 RGBA8 bricks (build-defined; EngineConfig.h:24-25 declares brick
// counts, no reference shader fills bricks). Texel (i, j, k) of the brick of
// node n at depth d, cell c (resolution 2^d) is the lattice point
// 2c + (i, j, k) in half-cell units: per channel the mean over the depth-d
// cells touching it ({c-1, c}, {c} or {c, c+1} per axis for i = 0, 1, 2;
// cells outside the grid count as zero) of their node colours, truncated.
// Cells are packed x | y << 10 | z << 20 (depth <= 10).

__device__ __forceinline__ uint32_t pack_cell(uint32_t x, uint32_t y, uint32_t z) { return x | (y << 10) | (z << 20); }

// Root children: slot s = z | x << 1 | y << 2 (octreeNodeFlag.comp:40).
__global__ void k_brick_root_cells(uint32_t* __restrict__ cells)
{
    const uint32_t s = threadIdx.x;
    if (s < 8u) cells[s] = pack_cell((s >> 1) & 1u, (s >> 2) & 1u, s & 1u);
}

// The 8 children of every subdivided node of one depth range.
__global__ __launch_bounds__(256) void k_brick_child_cells(const uint2* __restrict__ pool, uint32_t begin,
                                                           uint32_t num, uint32_t node_count,
                                                           uint32_t* __restrict__ cells)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= num) return;
    const uint32_t n = begin + i;
    const uint32_t child = pool[n].x & 0x7fffffffu;
    if (!child || child + 8u > node_count) return;
    const uint32_t cc = cells[n];
    const uint32_t x = 2u * (cc & 1023u), y = 2u * ((cc >> 10) & 1023u), z = 2u * (cc >> 20);
#pragma unroll
    for (uint32_t s = 0; s < 8u; ++s) cells[child + s] = pack_cell(x + ((s >> 1) & 1u), y + ((s >> 2) & 1u), z + (s & 1u));
}

// The depth's node colours into its dense grid (2^d cells per axis).
__global__ __launch_bounds__(256) void k_brick_scatter(const uint2* __restrict__ pool, const uint32_t* __restrict__ cells,
                                                       uint32_t begin, uint32_t num, uint32_t depth,
                                                       uint32_t* __restrict__ grid)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= num) return;
    const uint32_t n = begin + i, cc = cells[n], r = 1u << depth;
    const size_t at = ((size_t)(cc >> 20) * r + ((cc >> 10) & 1023u)) * r + (cc & 1023u);
    grid[at] = pool[n].y;
}

// RGBA8 -> four 16-bit lanes of a 64-bit word (sums of up to 8 bytes fit a lane).
__device__ __forceinline__ unsigned long long widen(uint32_t v)
{
    return (unsigned long long)(v & 0xffu) | ((unsigned long long)((v >> 8) & 0xffu) << 16) |
           ((unsigned long long)((v >> 16) & 0xffu) << 32) | ((unsigned long long)(v >> 24) << 48);
}

// Per-lane floor(lane / 2^sh), repacked to RGBA8. Every lane holds a sum of
// at most 2^sh bytes, so the quotient fits 8 bits; the mask keeps the next
// lane's low bits (shifted down into bits 16 - sh and up) out of it.
__device__ __forceinline__ uint32_t narrow(unsigned long long v, uint32_t sh)
{
    const unsigned long long m = 0xffull;
    return (uint32_t)(((v >> sh) & m) | (((v >> (16 + sh)) & m) << 8) | (((v >> (32 + sh)) & m) << 16) |
                      (((v >> (48 + sh)) & m) << 24));
}

__global__ __launch_bounds__(256) void k_brick_fill(const uint32_t* __restrict__ cells, uint32_t begin, uint32_t num,
                                                    uint32_t depth, const uint32_t* __restrict__ grid,
                                                    uint32_t* __restrict__ bricks)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= num) return;
    const uint32_t n = begin + i, cc = cells[n];
    const int r = 1 << depth;
    const int c[3] = {(int)(cc & 1023u), (int)((cc >> 10) & 1023u), (int)(cc >> 20)};
    // the 3x3x3 cells around c, widened, x fastest: v[dz][dy][dx] for d in {-1, 0, 1}
    unsigned long long v[27];
#pragma unroll
    for (int t = 0; t < 27; ++t) {
        const int x = c[0] + t % 3 - 1, y = c[1] + (t / 3) % 3 - 1, z = c[2] + t / 9 - 1;
        const bool in = x >= 0 && y >= 0 && z >= 0 && x < r && y < r && z < r;
        v[t] = in ? widen(grid[((size_t)z * (size_t)r + (size_t)y) * (size_t)r + (size_t)x]) : 0ull;
    }
    // separable sums: per axis texel 0 takes cells {-1, 0}, 1 takes {0}, 2 takes {0, +1}
    unsigned long long sx[27], sy[27];
#pragma unroll
    for (int zy = 0; zy < 9; ++zy) {
        sx[zy * 3 + 0] = v[zy * 3 + 0] + v[zy * 3 + 1];
        sx[zy * 3 + 1] = v[zy * 3 + 1];
        sx[zy * 3 + 2] = v[zy * 3 + 1] + v[zy * 3 + 2];
    }
#pragma unroll
    for (int z = 0; z < 3; ++z)
#pragma unroll
        for (int x = 0; x < 3; ++x) {
            sy[(z * 3 + 0) * 3 + x] = sx[(z * 3 + 0) * 3 + x] + sx[(z * 3 + 1) * 3 + x];
            sy[(z * 3 + 1) * 3 + x] = sx[(z * 3 + 1) * 3 + x];
            sy[(z * 3 + 2) * 3 + x] = sx[(z * 3 + 1) * 3 + x] + sx[(z * 3 + 2) * 3 + x];
        }
    uint32_t* out = bricks + 27u * (size_t)n;
#pragma unroll
    for (int y = 0; y < 3; ++y)
#pragma unroll
        for (int x = 0; x < 3; ++x) {
            const unsigned long long a = sy[(0 * 3 + y) * 3 + x], b = sy[(1 * 3 + y) * 3 + x], d = sy[(2 * 3 + y) * 3 + x];
            const uint32_t shxy = (uint32_t)(x != 1) + (uint32_t)(y != 1);
            out[(0 * 3 + y) * 3 + x] = narrow(a + b, shxy + 1u);
            out[(1 * 3 + y) * 3 + x] = narrow(b, shxy);
            out[(2 * 3 + y) * 3 + x] = narrow(b + d, shxy + 1u);
        }
}

// OctreeBuilder::cmdBuild (OctreeBuilder.cpp:205-345).
vct_status vct_svo_build(vct_ctx* c, vct_stream stream)
{
    if (!c) return fail(VCT_ERR_INVALID_ARGUMENT, "null context");
    if (!c->svo.level) return fail(VCT_ERR_NOT_READY, "vct_svo_voxelize has not run");
    hipStream_t s = (hipStream_t)stream;
    const uint32_t L = c->svo.level, R = 1u << L, nfrag = c->svo.nfrag;
    const bool half = (c->cfg.quirks & VCT_QUIRK_SVO_HALF_COORDS) != 0;
    // OctreeBuilder.cpp:110-113: clamp(8 * fragments, 1e6, 5e8) nodes
    uint64_t cap = (uint64_t)nfrag << 3;
    if (cap < 1000000ull) cap = 1000000ull;
    if (cap > 500000000ull) cap = 500000000ull;
    VCT_TRY(ensure(c->svo.pool, 8u * (size_t)cap));
    c->svo.pool_nodes = (uint32_t)cap;
    uint2* pool = (uint2*)c->svo.pool.ptr;
    const uint2* frags = (const uint2*)c->svo.frags.ptr;
    // sizes per depth, then the pool
    unsigned long long reached[kSvoMaxDepth] = {};  // nodes that some fragment reaches, but the leaves
    if (nfrag) {
        if (L <= 10) VCT_TRY(svo_sort<uint32_t>(c, s, frags, nfrag, L, half));
        else VCT_TRY(svo_sort<unsigned long long>(c, s, frags, nfrag, L, half));
        // the leaves' number is not needed: an octree of one level waits for nothing
        if (L > 1) {
            if (!c->pinned_word) VCT_HIP(hipHostMalloc(&c->pinned_word, kPinnedWordBytes, hipHostMallocDefault));
            VCT_HIP(hipMemcpyAsync(c->pinned_word, c->totals.ptr, 8u * (L - 1), hipMemcpyDeviceToHost, s));
            VCT_HIP(hipStreamSynchronize(s));
        }
        for (uint32_t e = 0; e + 1 < L; ++e) reached[e] = ((volatile unsigned long long*)c->pinned_word)[e];
    }
    // depth e's nodes: the eight of the root, then eight per node reached above
    std::vector<uint32_t> level_begin, level_num;
    uint64_t total = 0;
    for (uint32_t e = 0; e < L; ++e) {
        const uint64_t num = e ? 8ull * reached[e - 1] : 8ull;
        if (num == 0) break;  // no fragment: the tree ends here (the reference's zero-group dispatches)
        if (total + num > cap) return fail(VCT_ERR_CAPACITY, "octree node pool overflow (%llu nodes)", (unsigned long long)cap);
        level_begin.push_back((uint32_t)total);
        level_num.push_back((uint32_t)num);
        total += num;
    }
    // octreeNodeInit.comp
    hipLaunchKernelGGL(k_fill_u2, dim3(blocks_for(total)), dim3(256), 0, s, pool, (uint32_t)total, make_uint2(0u, 0u));
    if (nfrag) {
        if (L <= 10) svo_nodes<uint32_t>(c, s, nfrag, L, pool);
        else svo_nodes<unsigned long long>(c, s, nfrag, L, pool);
    }
    VCT_HIP(hipGetLastError());
    c->svo.node_count = (uint32_t)total;
    // octreeNodeMipmapWrite.comp for i = 2..L (OctreeBuilder.cpp:328-344). The
    // target of pass i is the node whose descent resolution equals i (quirk:
    // only i in {2, 4, 8} exist) or 2^(i-1); that node sits at depth
    // L - log2(target), whose pool range is level_begin/num of that depth.
    const bool quirk = (c->cfg.quirks & VCT_QUIRK_SVO_MIP_LEVEL_TEST) != 0;
    for (uint32_t i = 2; i <= L; ++i) {
        uint32_t target = quirk ? i : (1u << (i - 1));
        if (target & (target - 1)) continue;  // not a power of two: no node has that resolution
        uint32_t lg = 0;
        while ((1u << lg) < target) ++lg;
        if (lg >= L) continue;
        const uint32_t depth = L - lg;  // 1-based depth of the target nodes
        if (depth < 1 || depth > level_begin.size()) continue;
        hipLaunchKernelGGL(k_svo_mip, dim3(blocks_for(level_num[depth - 1])), dim3(256), 0, s, pool,
                           level_begin[depth - 1], level_num[depth - 1]);
    }
    // the octree trace's walk table
    c->svo.top_bits = L > kSvoTopBits ? L - kSvoTopBits : 0u;
    if (c->svo.top_bits) {
        const size_t cells = (size_t)1 << (3u * c->svo.top_bits);
        VCT_TRY(ensure(c->svo.top, sizeof(uint2) * cells));
        hipLaunchKernelGGL(k_svo_top, dim3(blocks_for(cells)), dim3(256), 0, s, (const uint2*)pool, L, c->svo.top_bits,
                           (uint2*)c->svo.top.ptr);
    }
    VCT_HIP(hipGetLastError());
    c->svo.depths = (uint32_t)level_begin.size();
    for (uint32_t d = 0; d < c->svo.depths; ++d) {
        c->svo.level_begin[d] = level_begin[d];
        c->svo.level_num[d] = level_num[d];
    }
    c->svo.built = true;
    c->svo.bricks_built = false;
    return VCT_OK;
}

vct_status vct_svo_build_bricks(vct_ctx* c, vct_stream stream)
{
    if (!c) return fail(VCT_ERR_INVALID_ARGUMENT, "null context");
    if (!c->svo.built) return fail(VCT_ERR_NOT_READY, "vct_svo_build has not run");
    const uint32_t L = c->svo.level;
    if (L > 10) return fail(VCT_ERR_UNSUPPORTED, "bricks are built for octree levels up to 10 (level %u)", L);
    hipStream_t s = (hipStream_t)stream;
    const uint32_t n = c->svo.node_count;
    size_t grid_total = 0;
    unsigned long long off[12] = {};
    for (uint32_t d = 1; d <= c->svo.depths; ++d) {
        off[d] = grid_total;
        grid_total += (size_t)1 << (3 * d);
    }
    VCT_TRY(ensure(c->svo.cells, 4u * (size_t)n));
    VCT_TRY(ensure(c->svo.grids, 4u * (grid_total ? grid_total : 1)));
    VCT_TRY(ensure(c->svo.bricks, 4u * 27u * (size_t)n));
    const uint2* pool = (const uint2*)c->svo.pool.ptr;
    uint32_t* cells = (uint32_t*)c->svo.cells.ptr;
    uint32_t* grids = (uint32_t*)c->svo.grids.ptr;
    VCT_HIP(hipMemsetAsync(grids, 0, 4u * grid_total, s));
    hipLaunchKernelGGL(k_brick_root_cells, dim3(1), dim3(64), 0, s, cells);
    for (uint32_t d = 1; d <= c->svo.depths; ++d) {
        const uint32_t b = c->svo.level_begin[d - 1], num = c->svo.level_num[d - 1];
        if (!num) continue;
        if (d < c->svo.depths)
            hipLaunchKernelGGL(k_brick_child_cells, dim3(blocks_for(num)), dim3(256), 0, s, pool, b, num, n, cells);
        hipLaunchKernelGGL(k_brick_scatter, dim3(blocks_for(num)), dim3(256), 0, s, pool, cells, b, num, d,
                           grids + off[d]);
    }
    for (uint32_t d = 1; d <= c->svo.depths; ++d) {
        const uint32_t b = c->svo.level_begin[d - 1], num = c->svo.level_num[d - 1];
        if (!num) continue;
        hipLaunchKernelGGL(k_brick_fill, dim3(blocks_for(num)), dim3(256), 0, s, (const uint32_t*)cells, b, num, d,
                           (const uint32_t*)(grids + off[d]), (uint32_t*)c->svo.bricks.ptr);
    }
    VCT_HIP(hipGetLastError());
    c->svo.bricks_built = true;
    return VCT_OK;
}

vct_status vct_svo_read_bricks(vct_ctx* c, vct_stream stream, uint32_t* out, size_t cap_bricks, size_t* n_bricks)
{
    if (!c || !n_bricks) return fail(VCT_ERR_INVALID_ARGUMENT, "null argument");
    if (!c->svo.bricks_built) return fail(VCT_ERR_NOT_READY, "vct_svo_build_bricks has not run");
    *n_bricks = c->svo.node_count;
    if (!out) return VCT_OK;
    if (cap_bricks < c->svo.node_count)
        return fail(VCT_ERR_CAPACITY, "output holds %zu bricks, the octree has %u", cap_bricks, c->svo.node_count);
    hipStream_t s = (hipStream_t)stream;
    VCT_HIP(hipMemcpyAsync(out, c->svo.bricks.ptr, 4u * 27u * (size_t)c->svo.node_count, hipMemcpyDeviceToHost, s));
    VCT_HIP(hipStreamSynchronize(s));
    return VCT_OK;
}

// OctreeBuilder::readOctreeNodes (OctreeBuilder.cpp:359-385): host copy of the
// allocated part of the pool (uvec2 per node).
vct_status vct_svo_read_nodes(vct_ctx* c, vct_stream stream, uint32_t* out, size_t cap_nodes, size_t* n_nodes)
{
    if (!c || !n_nodes) return fail(VCT_ERR_INVALID_ARGUMENT, "null argument");
    if (!c->svo.built) return fail(VCT_ERR_NOT_READY, "vct_svo_build has not run");
    *n_nodes = c->svo.node_count;
    if (!out) return VCT_OK;
    if (cap_nodes < c->svo.node_count) return fail(VCT_ERR_CAPACITY, "output holds %zu nodes, pool has %u", cap_nodes, c->svo.node_count);
    hipStream_t s = (hipStream_t)stream;
    VCT_HIP(hipMemcpyAsync(out, c->svo.pool.ptr, 8u * (size_t)c->svo.node_count, hipMemcpyDeviceToHost, s));
    VCT_HIP(hipStreamSynchronize(s));
    return VCT_OK;
}

// SparseVoxelizer::readVoxelFragments (SparseVoxelizer.cpp:328-353).
vct_status vct_svo_read_fragments(vct_ctx* c, vct_stream stream, uint32_t* out, size_t cap, size_t* n)
{
    if (!c || !n) return fail(VCT_ERR_INVALID_ARGUMENT, "null argument");
    *n = c->svo.nfrag;
    if (!out || !c->svo.nfrag) return VCT_OK;
    if (cap < c->svo.nfrag) return fail(VCT_ERR_CAPACITY, "output holds %zu fragments, list has %u", cap, c->svo.nfrag);
    hipStream_t s = (hipStream_t)stream;
    VCT_HIP(hipMemcpyAsync(out, c->svo.frags.ptr, 8u * (size_t)c->svo.nfrag, hipMemcpyDeviceToHost, s));
    VCT_HIP(hipStreamSynchronize(s));
    return VCT_OK;
}

// Device pointer to the node pool ("OctreeBuilder::getOctreeBuffer").
vct_status vct_svo_pool(vct_ctx* c, const uint32_t** pool, uint32_t* node_count)
{
    if (!c || !pool || !node_count) return fail(VCT_ERR_INVALID_ARGUMENT, "null argument");
    if (!c->svo.built) return fail(VCT_ERR_NOT_READY, "vct_svo_build has not run");
    *pool = (const uint32_t*)c->svo.pool.ptr;
    *node_count = c->svo.node_count;
    return VCT_OK;
}

}  // extern "C"
