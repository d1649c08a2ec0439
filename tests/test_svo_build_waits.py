"""The host's waits in the octree build: one read-back of the depths' sizes, and
none for an octree of one level, whose eight nodes are known. The library's host
code against a stand-in for the HIP runtime."""
import subprocess

import pytest

import hip_stand_in

MAIN = r"""
int main(int, char** argv)
{
    void* lib = dlopen(argv[1], RTLD_LAZY | RTLD_LOCAL);
    if (!lib) { fprintf(stderr, "%s\n", dlerror()); return 9; }
    vct_config cfg{16, 1, VCT_FORMAT_RGBA8, 0, 1, 1, 1.0f, 0};
    vct_ctx* c = nullptr;
    if (CALL(vct_create)(&c, &cfg) != VCT_OK) return 8;
    static float img[4], zero[32];
    static uint32_t index[3];
    vct_shadow_map shadow{img, 1, 1};
    vct_directional_light_desc light{};
    vct_directional_light_shadow_desc light_shadow{};
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
    for (int k = 0; k < 3; ++k) mesh.scene_bb_max[k] = 1.0f;
    counted = 1;  // one work item, one fragment
    uint32_t n = 0;
    if (CALL(vct_svo_voxelize)(c, nullptr, &mesh, &shadow, &light, &light_shadow, atoi(argv[2]), &n) != VCT_OK || n != 1)
        return 7;
    waits = 0;
    launched.clear();
    const vct_status s = CALL(vct_svo_build)(c, nullptr);
    printf("%d %d %s\n", (int)s, waits, launched.c_str());
    return 0;
}
"""


@pytest.mark.parametrize("level,waits", [(1, 0), (2, 1), (9, 1)])
def test_build_waits(level, waits, tmp_path):
    from vk_voxel_cone_tracing_amd import _abi

    host = hip_stand_in.build(tmp_path, MAIN)
    r = subprocess.run([host, str(_abi.LIB_PATH), str(level)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stderr)
    status, got, kernels = r.stdout.split(" ", 2)
    assert int(status) == 0 and "k_svo_nodes" in kernels
    assert int(got) == waits, r.stdout
