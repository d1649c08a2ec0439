"""The dense mip tail (dense_mip_tail in csrc/vct_dense_mip.hpp) stays inside
its LDS array: the header, compiled for the host with AddressSanitizer and the
array as a local one, at every resolution whose tail starts at another level.
Its levels are compared with dense_mip_texel_lean's, face by face."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vk_voxel_cone_tracing_amd", "csrc")

STUB = """#pragma once
#include <cstddef>
#include <cstdint>
#define __device__
#define __host__
#define __forceinline__ inline
#define __shared__  // a local array: one thread is the whole workgroup
#define _Float16 short  // the half texels are not used here
struct float4 { float x, y, z, w; };
struct uint2 { unsigned x, y; };
inline float4 make_float4(float x, float y, float z, float w) { return {x, y, z, w}; }
typedef void* hipStream_t;
typedef int hipError_t;
static const struct { unsigned x; } threadIdx = {0}, blockDim = {1};
inline void __syncthreads() {}
inline float __builtin_amdgcn_fmed3f(float f, float lo, float hi) { return f > lo ? (f < hi ? f : hi) : lo; }
"""

MAIN = r"""
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>
#include "vct_dense_mip.hpp"
using namespace vct;

template <bool kF32>
static int run(int res)
{
    const size_t texel = kF32 ? 16 : 4;
    unsigned long long offset[11];
    size_t texels = 0;
    int nlevels = 0;
    for (int n = res; n >= 1; n /= 2, ++nlevels) {
        offset[nlevels] = texels;
        texels += dense_mip_block(n) * (nlevels ? kFaces : 1);
    }
    std::vector<char> got(texels * texel), want(texels * texel);
    std::mt19937 rng(res);
    for (int z = 0; z < res; ++z)
        for (int y = 0; y < res; ++y)
            for (int x = 0; x < res; ++x) {
                auto u = [&] { return std::uniform_real_distribution<float>(0.0f, 1.0f)(rng); };
                dense_store<kF32>(want.data(), dense_mip_index(res, x, y, z), f4{u(), u(), u(), u()});
            }
    int first = 1;  // the first level of the tail
    while (first < nlevels && (res >> first) > tail_edge<kF32>()) ++first;
    for (int m = 1; m < nlevels; ++m) {
        if (m == first) memcpy(got.data(), want.data(), offset[m] * texel);
        const int n = res >> m;
        for (int z = 0; z < n; ++z)
            for (int y = 0; y < n; ++y)
                for (int x = 0; x < n; ++x)
                    dense_mip_texel_lean<kF32>(&want[offset[m - 1] * texel], &want[offset[m] * texel], n, x, y, z, m == 1);
    }
    for (int f = 0; f < kFaces; ++f) dense_mip_tail<kF32>(got.data(), offset, res, first, nlevels, f);
    return memcmp(got.data(), want.data(), got.size()) != 0;
}

int main(int, char** argv)
{
    const int res = atoi(argv[2]);
    return atoi(argv[1]) ? run<true>(res) : run<false>(res);
}
"""


@pytest.fixture(scope="module")
def tail(tmp_path_factory):
    d = tmp_path_factory.mktemp("tail")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(STUB)
    (d / "main.cpp").write_text(MAIN)
    exe = str(d / "tail")
    subprocess.run(["g++", "-std=c++17", "-O1", "-ffp-contract=off", "-w", "-fsanitize=address", f"-I{d}", f"-I{CSRC}",
                    str(d / "main.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("f32", [0, 1])
@pytest.mark.parametrize("res", [2, 4, 8, 16, 32, 64])
def test_tail_stays_inside_its_array(tail, f32, res):
    # a preloaded library may come before the sanitizer's own
    env = dict(os.environ, ASAN_OPTIONS="verify_asan_link_order=0")
    r = subprocess.run([tail, str(f32), str(res)], capture_output=True, text=True, env=env)
    assert r.returncode == 0, r.stderr[:2000]
