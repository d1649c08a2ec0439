"""The cell range of a triangle (tri_setup in csrc/vct_raster.hpp) holds every
covered sample: the header, compiled for the host, against all samples of the
bounding box and six cells around it. Triangles of every size from a hundredth
of a voxel to hundreds, slivers down to a few units in the last place, edges on
cell and sample lines, coordinates far from the origin and tiny ones."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vk_voxel_cone_tracing_amd", "csrc")

STUB = """#pragma once
#include <algorithm>
#include <cmath>
#define __device__
#define __constant__
#define __forceinline__ inline
using std::max;
using std::min;
"""

MAIN = r"""
#include <cstdio>
#include <cstdlib>
#include <random>
#include "vct_raster.hpp"
using namespace vct;
int main(int argc, char** argv)
{
    const int samples = atoi(argv[1]);
    std::mt19937 rng(samples);
    auto uni = [&](float a, float b) { return std::uniform_real_distribution<float>(a, b)(rng); };
    const int lo[3] = {-200000, -200000, -200000}, hi[3] = {200000, 200000, 200000};
    long covered = 0, items = 0, general = 0;
    for (int k = 0; k < 60000; ++k) {
        const float vs = k % 3 == 0 ? 0.25f : (k % 3 == 1 ? 2.0f / 511.0f : uni(0.001f, 3.0f));
        const float size = vs * std::pow(10.0f, uni(-2.0f, k % 50 ? 0.9f : 1.6f));
        const int form = k % 8;
        float at[3], p[9];
        for (int j = 0; j < 3; ++j) at[j] = form == 7 ? uni(-1e4f, 1e4f) * vs : uni(-3.0f, 3.0f) * vs;
        if (form == 6) for (int j = 0; j < 3; ++j) at[j] = uni(-1.0f, 1.0f) * (k % 16 == 6 ? 1e-12f : 60000.0f * vs);
        for (int j = 0; j < 9; ++j) p[j] = at[j % 3] + uni(-1.0f, 1.0f) * size;
        if (form == 1)  // slivers: the third vertex on the first edge but for rounding
            for (int j = 0; j < 3; ++j) p[6 + j] = p[j] + (p[3 + j] - p[j]) * uni(-1.0f, 2.0f);
        if (form == 2)  // thin
            for (int j = 0; j < 3; ++j) p[6 + j] = p[j] + (p[3 + j] - p[j]) * 0.5f + uni(-1e-3f, 1e-3f) * size;
        if (form == 3)  // vertices on the lines of cells and samples
            for (int j = 0; j < 9; ++j) p[j] = std::round(p[j] / vs * 8.0f) / 8.0f * vs;
        if (form == 4)  // axis-aligned
            for (int j = 0; j < 9; ++j) p[j] = std::round(p[j] / vs) * vs + 0.5f * vs * (j % 2);
        TriSetup s{}, all;
        const bool any = tri_setup(p, vs, samples, lo, hi, s);
        // s holds the edges either way, unless the triangle has no area
        if (s.area == 0.0 && !any) continue;
        all = s;
        float umin = std::min({p[s.u], p[3 + s.u], p[6 + s.u]}), umax = std::max({p[s.u], p[3 + s.u], p[6 + s.u]});
        float vmin = std::min({p[s.v], p[3 + s.v], p[6 + s.v]}), vmax = std::max({p[s.v], p[3 + s.v], p[6 + s.v]});
        all.cu_lo = (int)std::floor(umin / vs) - 6;
        all.cv_lo = (int)std::floor(vmin / vs) - 6;
        all.nu = (int)std::floor(umax / vs) + 6 - all.cu_lo + 1;
        all.nv = (int)std::floor(vmax / vs) + 6 - all.cv_lo + 1;
        general += (long)(all.nu - 8) * (all.nv - 8);
        if (any) items += (long)s.nu * s.nv;
        for (uint32_t i = 0; i < (uint32_t)(all.nu * all.nv * samples); ++i) {
            float pos[3];
            double lam[3];
            if (!tri_sample(p, all, vs, samples, i, pos, lam)) continue;
            ++covered;
            const int cu = all.cu_lo + (int)(i / samples) % all.nu, cv = all.cv_lo + (int)(i / samples) / all.nu;
            if (!any || cu < s.cu_lo || cu >= s.cu_lo + s.nu || cv < s.cv_lo || cv >= s.cv_lo + s.nv) {
                // the general range (one cell around the box) holds no more than this either
                const int gu = (int)std::floor(umin / vs) - 1, gv = (int)std::floor(vmin / vs) - 1;
                const int hu = (int)std::floor(umax / vs) + 1, hv = (int)std::floor(vmax / vs) + 1;
                if (cu < gu || cu > hu || cv < gv || cv > hv) continue;
                printf("triangle %d form %d: covered cell (%d, %d) outside\n", k, form, cu, cv);
                return 1;
            }
        }
    }
    printf("%ld covered, %ld cells in range, %ld around the boxes\n", covered, items, general);
    return covered > 100000 && items < general ? 0 : 2;
}
"""


@pytest.mark.parametrize("samples", [1, 4])
def test_range_holds_every_covered_sample(samples, tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(STUB)
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = str(tmp_path / "range")
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-w", f"-I{tmp_path}", f"-I{CSRC}", str(tmp_path / "main.cpp"),
                    "-o", exe], check=True)
    r = subprocess.run([exe, str(samples)], capture_output=True, text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
