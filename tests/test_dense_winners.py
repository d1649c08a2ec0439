"""The winners of the dense voxelizer are kept empty from one call to the next:
filled by the first call, by the call after one that failed, and by every call
after a fill that was only recorded into a graph. A host program stands in for
the HIP runtime (its symbols come before the library's), so that no kernel
runs, any launch can be made to fail, and the launches of a call are listed."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]

MAIN = r"""
#include <dlfcn.h>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include "vct.h"

// ---- the HIP runtime, on host memory
struct dim3 { unsigned x, y, z; };
static std::map<const void*, std::string> names;
static std::string launched, failing;
static int last_error = 0, capturing = 0;
static dim3 grid_, block_;
static size_t shared_;
static void* stream_;
extern "C" {
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*)
{
    names[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t m, void* s) { grid_ = g; block_ = b; shared_ = m; stream_ = s; return 0; }
int __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, void** s) { *g = grid_; *b = block_; *m = shared_; *s = stream_; return 0; }
int hipLaunchKernel(const void* f, dim3, dim3, void**, size_t, void*)
{
    const std::string& n = names[f];
    if (!failing.empty() && n.find(failing) != std::string::npos) return last_error = 1;
    launched += n + ' ';
    return 0;
}
int hipGetLastError() { const int e = last_error; last_error = 0; return e; }
const char* hipGetErrorString(int) { return "error"; }
int hipMalloc(void** p, size_t n) { return (*p = calloc(1, n)) ? 0 : 2; }
int hipFree(void* p) { free(p); return 0; }
int hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
int hipHostFree(void* p) { return hipFree(p); }
int hipMemset(void* p, int v, size_t n) { memset(p, v, n); return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) { memcpy(d, s, n); return 0; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipDeviceSynchronize() { return 0; }
int hipStreamSynchronize(void*) { return 0; }
int hipGetSymbolAddress(void** p, const void*) { static char c; *p = &c; return 0; }
int hipStreamIsCapturing(void*, int* s) { *s = capturing; return 0; }
}

#define CALL(name) ((decltype(&name))dlsym(lib, #name))

int main(int, char** argv)
{
    void* lib = dlopen(argv[1], RTLD_LAZY | RTLD_LOCAL);
    if (!lib) { fprintf(stderr, "%s\n", dlerror()); return 9; }
    vct_dense_desc d{};
    d.extent = 1.0f;
    d.resolution = 8;
    d.format = VCT_FORMAT_RGBA8;
    d.raster_samples = 1;
    float zero[32] = {};
    uint32_t index[3] = {};
    vct_gltf_material mat{};
    mat.base_color_texture = mat.emissive_texture = mat.occlusion_texture = -1;
    vct_primitive prim{};
    prim.index_count = 3;
    vct_mesh mesh{};
    mesh.positions = mesh.normals = mesh.node_matrices = zero;
    mesh.indices = index;
    mesh.materials = &mat;
    mesh.vertex_count = mesh.instance_count = mesh.material_count = mesh.primitive_count = 1;
    mesh.index_count = 3;
    mesh.primitives = &prim;
    vct_dense* g = nullptr;
    if (CALL(vct_dense_create)(&g, &d) != VCT_OK) return 8;
    // one call: whether it succeeds, and whether it fills the winners
    auto voxelize = [&](bool ok, bool fills, const char* what) {
        launched.clear();
        const bool done = CALL(vct_dense_voxelize)(g, nullptr, &mesh) == VCT_OK;
        const bool filled = launched.find("k_fill_u32") != std::string::npos;
        if (done != ok || filled != fills) {
            printf("%s: %s, winners %sfilled [%s]\n", what, done ? "done" : "failed", filled ? "" : "not ", launched.c_str());
            exit(1);
        }
    };
    if (!argv[2][0]) {  // a first call that is only recorded
        capturing = 1;
        voxelize(true, true, "recorded");
        capturing = 0;
        voxelize(true, true, "first after the recording");
        voxelize(true, false, "second after the recording");
        capturing = 1;
        voxelize(true, false, "recorded with the winners empty");
        capturing = 0;
        voxelize(true, false, "after it");
        return 0;
    }
    failing = argv[2];
    const bool fill = failing == "k_fill_u32";
    if (!fill) {
        failing.clear();
        voxelize(true, true, "first");
        voxelize(true, false, "second");
        failing = argv[2];
    }
    voxelize(false, false, "failing");
    failing.clear();
    voxelize(true, true, "after the failure");
    voxelize(true, false, "and the next");
    return 0;
}
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    d = tmp_path_factory.mktemp("winners")
    (d / "main.cpp").write_text(MAIN)
    exe = str(d / "host")
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-rdynamic", f"-I{ROOT / 'include'}", str(d / "main.cpp"), "-ldl",
                    "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("failing", ["k_fill_u32", "k_dense_count", "k_dense_total", "k_dense_raster", "k_dense_resolve",
                                     ""])
def test_winners_are_filled_after_a_failure(host, failing):
    from vk_voxel_cone_tracing_amd import _abi

    r = subprocess.run([host, str(_abi.LIB_PATH), failing], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
