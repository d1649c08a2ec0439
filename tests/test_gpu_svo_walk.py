"""The octree trace's walks against the oracle: octrees too small for the walk
table (5 levels), with a table of 2^3 and 8^3 cells, and a table that does not
serve the trace (volume_dimension other than the octree's); sixteen and four
waves per tile, 16 and 32 cones, and a view that looks out of the scene box."""
import ctypes as C

import numpy as np
import pytest

import oracle_api as O
import test_gpu_svo as svo

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level,dim,cones32,W,H", [(5, 32, 0, 33, 17), (6, 64, 1, 200, 120), (8, 256, 0, 61, 40),
                                                   (8, 64, 0, 61, 40)])
def test_walks_match_oracle(level, dim, cones32, W, H):
    import torch
    import vk_voxel_cone_tracing_amd as V
    from vk_voxel_cone_tracing_amd import scenes

    r = svo._run(0x00, level=level)
    scene = r["scene"]
    vp, vp_inv, eye = scenes.camera(3, W, H, scale=1.0)
    g = O.raycast_gbuffer(scene, r["pos"], r["nrm"], r["mat"], vp, vp_inv, W, H)
    views = {np.dtype(np.uint32): np.int32, np.dtype(np.uint16): np.int16}
    gd = {k: torch.from_numpy(v.view(views.get(v.dtype, v.dtype))).cuda() for k, v in g.items()}
    vs, center = 1.0 / dim, [0.5, 0.5, 0.5]
    desc = V._abi.ConeTracingDesc(V._abi.f3(*center), 8, vs, float(dim), 1.0, 8.0, 0.5, 1.0, 3.0, 2.0, cones32)
    dout = torch.zeros((H, W, 4), device="cuda")
    sout = torch.zeros_like(dout)
    lo, hi = (C.c_float * 3)(*scene.bb_min.tolist()), (C.c_float * 3)(*scene.bb_max.tolist())
    V._abi.call("vct_svo_trace", r["ctx"]._h, None, C.byref(V.gbuffer_struct(gd)),
                C.byref(V.camera_ubo(vp, vp_inv, eye)), C.byref(desc), C.byref(r["sm"]), C.byref(r["ld"]),
                C.byref(r["ls"]), lo, hi, C.c_void_p(dout.data_ptr()), C.c_void_p(sout.data_ptr()), None)
    torch.cuda.synchronize()
    fields = dict(volume_center=center, rendering_mode=8, voxel_size=vs, volume_dimension=float(dim),
                  trace_start_offset=1.0, indirect_diffuse_intensity=8.0, ambient_occlusion_factor=0.5,
                  min_trace_step_factor=1.0, indirect_specular_intensity=3.0, occlusion_decay=2.0,
                  enable_32_cones=cones32)
    p = O.trace_params(fields, vp_inv, eye, 6)
    rd, rs = np.zeros((H, W, 4), np.float32), np.zeros((H, W, 4), np.float32)
    osm = O.Shadow(r["depth"].ctypes.data, 128, 128)
    O.lib().orc_svo_trace(O.vptr(np.ascontiguousarray(r["onodes"])), C.byref(O.gbuf_struct(g)), C.byref(p), lo, hi,
                          C.byref(osm), C.byref(O.light_struct(r["light"])), 0x00, 0, H, O.vptr(rd), O.vptr(rs), None)
    # a sample whose position rounds across a cell face reads another node: the
    # bound of the octree trace's own oracle test
    for name, got, ref in (("diffuse", dout.cpu().numpy(), rd), ("specular", sout.cpu().numpy(), rs)):
        err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
        print(f"level {level} dim {dim} {name}: rel L2 {err:.2e}")
        assert err <= 1e-3, (name, err)
