"""The traces of images above the sizes that are split (more than 8192 tiles of
8x8 pixels: one wave per tile; more than 2^19 pixels: one lane per specular
cone): a whole 1030x530 image with edge tiles cut on both sides, its first,
middle and last rows against the oracle. And several views whose tiles only
together pass the line, against one call per view, which splits its tiles."""
import ctypes as C

import numpy as np
import pytest

import oracle_api as O
import test_gpu_clipmap as clipmap
import test_gpu_dense as dense
import test_gpu_dense_views as dense_views
import test_gpu_svo as svo

pytestmark = pytest.mark.gpu

W, H = 1030, 530
ROWS = (0, 1, 263, 264, 528, 529)


def _gbuffer(scene, ds, cam):
    """The device's G-buffer of the whole image, and its host copy."""
    import vk_voxel_cone_tracing_amd as V
    from vk_voxel_cone_tracing_amd import workloads

    sc = workloads.scratch_ctx()
    gd = workloads.gbuffer(sc, ds, scene, cam, W, H)
    V._abi.call("vct_destroy", sc)
    as_unsigned = {np.dtype(np.int32): np.uint32, np.dtype(np.int16): np.uint16}
    host = {k: v.cpu().numpy() for k, v in gd.items()}
    return gd, {k: v.view(as_unsigned.get(v.dtype, v.dtype)) for k, v in host.items()}


def _check(name, got, ref):
    rows = list(ROWS)
    err = np.linalg.norm(got[rows] - ref[rows]) / max(np.linalg.norm(ref[rows]), 1e-12)
    print(f"{name}: rel L2 {err:.2e}")
    # the bound of the smaller images' tests
    assert np.linalg.norm(ref[rows]) > 0 and err <= 1e-3, (name, err)


@pytest.mark.parametrize("fmt,mode,cones32", [(0, 8, 0), (0, 5, 1), (1, 7, 0)])
def test_clipmap_trace(fmt, mode, cones32):
    import torch
    import vk_voxel_cone_tracing_amd as V
    from vk_voxel_cone_tracing_amd import scenes

    res, levels = 32, 3
    scene, ctx, ds = clipmap._setup_case(0x3F, fmt=fmt, res=res, levels=levels)
    pos, nrm, mat = scene.world_triangles()
    light, depth, depth_d = clipmap._light_and_shadow(scene, pos, nrm, mat)
    (ld, ls), sm = V.light_structs(light), V.shadow_struct(depth_d)
    clipmap._pipeline(ctx, ds, scene, sm, ld, ls, levels)
    cam = scenes.camera(0, W, H, scale=clipmap.SCALE)
    gd, g = _gbuffer(scene, ds, cam)
    lo, n, vs = ctx.regions[0]
    center = [float(np.float32(lo[k] * vs + n[k] * vs * 0.5)) for k in range(3)]
    desc = V._abi.ConeTracingDesc(V._abi.f3(*center), mode, vs, float(res), 1.0, 8.0, 0.5, 1.0, 3.0, 2.0, cones32)
    dout = torch.zeros((H, W, 4), device="cuda")
    sout = torch.zeros_like(dout)
    ctx.trace(V.gbuffer_struct(gd), V.camera_ubo(*cam), desc, sm, ld, ls, dout, sout)
    torch.cuda.synchronize()
    fields = dict(volume_center=center, rendering_mode=mode, voxel_size=vs, volume_dimension=float(res),
                  trace_start_offset=1.0, indirect_diffuse_intensity=8.0, ambient_occlusion_factor=0.5,
                  min_trace_step_factor=1.0, indirect_specular_intensity=3.0, occlusion_decay=2.0,
                  enable_32_cones=cones32)
    rd, rs, _ = O.trace_rows(ctx.read_volume(V.VOLUME_RADIANCE), res, levels, g,
                             O.trace_params(fields, cam[1], cam[2], levels), depth, light, ROWS)
    _check(f"clipmap fmt={fmt} mode={mode} diffuse", dout.cpu().numpy(), rd)
    _check(f"clipmap fmt={fmt} mode={mode} specular", sout.cpu().numpy(), rs)


def test_octree_trace():
    import torch
    import vk_voxel_cone_tracing_amd as V
    from vk_voxel_cone_tracing_amd import scenes

    level, dim = 7, 128
    r = svo._run(0x00, level=level)
    scene, cam = r["scene"], scenes.camera(3, W, H, scale=1.0)
    gd, g = _gbuffer(scene, r["ds"], cam)
    vs, center = 1.0 / dim, [0.5, 0.5, 0.5]
    desc = V._abi.ConeTracingDesc(V._abi.f3(*center), 8, vs, float(dim), 1.0, 8.0, 0.5, 1.0, 3.0, 2.0, 0)
    dout = torch.zeros((H, W, 4), device="cuda")
    sout = torch.zeros_like(dout)
    lo, hi = (C.c_float * 3)(*scene.bb_min.tolist()), (C.c_float * 3)(*scene.bb_max.tolist())
    V._abi.call("vct_svo_trace", r["ctx"]._h, None, C.byref(V.gbuffer_struct(gd)), C.byref(V.camera_ubo(*cam)),
                C.byref(desc), C.byref(r["sm"]), C.byref(r["ld"]), C.byref(r["ls"]), lo, hi,
                C.c_void_p(dout.data_ptr()), C.c_void_p(sout.data_ptr()), None)
    torch.cuda.synchronize()
    fields = dict(volume_center=center, rendering_mode=8, voxel_size=vs, volume_dimension=float(dim),
                  trace_start_offset=1.0, indirect_diffuse_intensity=8.0, ambient_occlusion_factor=0.5,
                  min_trace_step_factor=1.0, indirect_specular_intensity=3.0, occlusion_decay=2.0, enable_32_cones=0)
    p = O.trace_params(fields, cam[1], cam[2], 6)
    rd, rs = np.zeros((H, W, 4), np.float32), np.zeros((H, W, 4), np.float32)
    osm = O.Shadow(r["depth"].ctypes.data, 128, 128)
    pool, gb, ol = np.ascontiguousarray(r["onodes"]), O.gbuf_struct(g), O.light_struct(r["light"])
    for row in ROWS:
        O.lib().orc_svo_trace(O.vptr(pool), C.byref(gb), C.byref(p), lo, hi, C.byref(osm), C.byref(ol), 0x00, row,
                              row + 1, O.vptr(rd), O.vptr(rs), None)
    _check("octree diffuse", dout.cpu().numpy(), rd)
    _check("octree specular", sout.cpu().numpy()[..., :3], rs[..., :3])


@pytest.mark.parametrize("fmt", [O.FMT_RGBA8, O.FMT_RGBA32F])
def test_dense_trace(fmt):
    import torch
    import vk_voxel_cone_tracing_amd as V
    from vk_voxel_cone_tracing_amd import scenes

    res = 64
    scene, h, grid_min, ext = dense._grid(fmt, res, 1)
    ds, cam = V.DeviceScene(scene), scenes.camera(5, W, H, scale=dense.SCALE)
    gd, g = _gbuffer(scene, ds, cam)
    td = V._abi.DenseTraceDesc(0.872665, 0.75 * ext, 1.0, 1.0, 2.0, 0.5, 8.0, 0)
    try:
        V._abi.call("vct_dense_voxelize", h, None, C.byref(ds.mesh))
        V._abi.call("vct_dense_mipmap", h, None)
        out = torch.zeros((H, W, 4), device="cuda")
        V._abi.call("vct_dense_trace", h, None, C.byref(V.gbuffer_struct(gd)), C.byref(V.camera_ubo(*cam)), C.byref(td),
                    C.c_void_p(out.data_ptr()), None)
        torch.cuda.synchronize()
        levels = dense._read_levels(h, res, fmt)
    finally:
        V._abi.call("vct_dense_destroy", h)
    d, ref = O.new_dense(res, fmt, grid_min, ext)
    for a, b in zip(ref, levels):
        a[...] = b
    p = O.dense_params(cam[1], aperture=td.aperture, max_dist=td.max_distance, decay=2.0, ao_factor=0.5,
                       diffuse_intensity=8.0)
    r64, gb = np.zeros((H, W, 4), np.float64), O.gbuf_struct(g)
    for row in ROWS:
        O.lib().orc_dense_trace(C.byref(d), C.byref(gb), C.byref(p), row, row + 1, O.vptr(r64), None)
    got = out.cpu().numpy().astype(np.float64)
    _check("dense indirect", got[..., :3], r64[..., :3])
    _check("dense ao", got[..., 3:], r64[..., 3:])


def test_dense_views_together_above_the_line():
    # 2176 tiles a view: four waves per tile alone, one in the call of four views
    dense_views.test_views_equal_single_calls(512, 270, 4, 0)
