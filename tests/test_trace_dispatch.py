"""How many waves the clipmap and octree traces put on a tile, by image size and
mode: the split over four and sixteen waves is for the diffuse cones, so the
modes that march none (the G-buffer views and the specular one) keep one wave
per tile at every size. The library's host code against a stand-in for the HIP
runtime; the waves are a template argument in the kernels' names."""
import re
import subprocess

import pytest

import hip_stand_in

MAIN = r"""
int main(int, char** argv)
{
    void* lib = dlopen(argv[1], RTLD_LAZY | RTLD_LOCAL);
    if (!lib) { fprintf(stderr, "%s\n", dlerror()); return 9; }
    vct_config cfg{16, 2, (uint32_t)atoi(argv[2]), 0, 1, 1, 1.0f, 0};
    vct_ctx* c = nullptr;
    if (CALL(vct_create)(&c, &cfg) != VCT_OK) return 8;
    static float img[4], zero[32];
    static uint32_t index[3];
    static uint16_t half[4];
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
    uint32_t n;
    if (CALL(vct_svo_voxelize)(c, nullptr, &mesh, &shadow, &light, &light_shadow, 4, &n) != VCT_OK) return 7;
    if (CALL(vct_svo_build)(c, nullptr) != VCT_OK) return 6;
    const unsigned sizes[4][2] = {{160, 90}, {640, 360}, {960, 540}, {1280, 720}};
    for (auto& s : sizes)
        for (unsigned mode = 0; mode < 9; ++mode) {
            vct_gbuffer g{};
            g.diffuse = g.specular = index;
            g.normal = g.emission = half;
            g.depth = img;
            g.width = s[0];
            g.height = s[1];
            vct_camera_ubo cam{};
            vct_cone_tracing_desc d{};
            d.rendering_mode = mode;
            d.voxel_size = 0.1f;
            d.volume_dimension = 16.0f;
            launched.clear();
            if (CALL(vct_trace)(c, nullptr, &g, &cam, &d, &shadow, &light, &light_shadow, img, img, nullptr) != VCT_OK)
                return 5;
            printf("clipmap %u %u %u %s\n", s[0], s[1], mode, launched.c_str());
            launched.clear();
            if (CALL(vct_svo_trace)(c, nullptr, &g, &cam, &d, &shadow, &light, &light_shadow, mesh.scene_bb_min,
                                    mesh.scene_bb_max, img, img, nullptr) != VCT_OK)
                return 4;
            printf("octree %u %u %u %s\n", s[0], s[1], mode, launched.c_str());
        }
    return 0;
}
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    return hip_stand_in.build(tmp_path_factory.mktemp("dispatch"), MAIN)


@pytest.mark.parametrize("fmt", [0, 1])
def test_waves_per_tile(host, fmt):
    from vk_voxel_cone_tracing_amd import _abi

    r = subprocess.run([host, str(_abi.LIB_PATH), str(fmt)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stderr)
    lines = r.stdout.splitlines()
    assert len(lines) == 2 * 4 * 9
    for line in lines:
        kind, w, h, mode, kernels = line.split(" ", 4)
        w, h, mode = int(w), int(h), int(mode)
        waves = [int(k) for k in re.findall(r"k_traceILb[01]ELb[01]ELi(\d+)E" if kind == "clipmap" else
                                            r"k_svo_traceILi(\d+)E", kernels)]
        tiles = 4 * ((w + 15) // 16) * ((h + 15) // 16)
        split = 16 if tiles <= 256 else 4 if tiles <= 8192 else 1
        assert waves == [split if mode in (4, 5, 7, 8) else 1], line
