"""The measured cases of the voxel cone tracing framework: what a program of
its users runs per frame, per build or per training step, through the public
entry points (Context, the render passes, the vct_* calls and adjoint.render).

Kinds of case (`kind`):
  frame    one clipmap GI frame: voxelization, radiance injection, cone trace
  moving   four frames of a moving camera: toroidal revoxelization, the clip
           levels due at each frame, cone trace
  baked    the cone trace alone over a clipmap the program wrote itself
  dense    the plain method: clear, voxelize, mips, ambient-occlusion trace
  svo      sparse voxel octree: fragments, pool, octree cone trace
  batch    many dense scenes replayed from one captured launch
  adjoint  one training step: differentiable render, loss, backward
  filter   the specular filter and tonemap after the trace

Inputs are seeded and synthetic: the procedural room of this package, or an
analytic room (walls and spheres) where the float64 reference needs one.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import vk_voxel_cone_tracing_amd as V
from vk_voxel_cone_tracing_amd import _abi as A
from vk_voxel_cone_tracing_amd import passes, scenes, workloads

SCALE = 16.0  # world edge of the room in the clipmap cases: clip level 0 spans it
QUIRK_CLAMP_X_RANGE = 1
MOVING_FRAMES = 4


def listed():
    return [
        # the flagship frame: 6 x 128^3 half-float clipmap at full HD
        dict(name="frame_1080p", kind="frame", W=1920, H=1080, res=128, levels=6, half=True, cones32=False, samples=1,
             shadow=2048, ao=False),
        # the reference's RGBA8 radiance at a ragged window size, 32 cones, 4 raster samples
        dict(name="frame_rgba8_32cones", kind="frame", W=1283, H=717, res=64, levels=5, half=False, cones32=True,
             samples=4, shadow=1024, ao=False),
        # a preview or probe: the smallest frame, bound by launches and latency
        dict(name="frame_160x90", kind="frame", W=160, H=90, res=32, levels=3, half=False, cones32=False, samples=1,
             shadow=512, ao=False),
        # a walk through the scene: slabs revoxelized, levels injected in turn
        dict(name="moving_camera", kind="moving", W=640, H=360, res=64, levels=4, half=True, shadow=1024),
        # a baked clipmap traced every frame
        dict(name="baked_trace", kind="baked", W=640, H=360, res=64, levels=4, half=True, cones32=False, shadow=512),
        # plain VXAO as the tests and the benchmark use it
        dict(name="dense_vxao_360p", kind="dense", W=640, H=360, res=128, tris=21260, cones32=False, samples=1),
        # a detailed scene in a large grid
        dict(name="dense_vxao_256", kind="dense", W=1021, H=768, res=256, tris=300000, cones32=False, samples=1),
        # octree rebuilt from a detailed mesh, then traced
        dict(name="svo_512", kind="svo", W=640, H=360, level=9, tris=1000000, shadow=2048),
        # many uneven scenes at once
        dict(name="batch_16", kind="batch", W=256, H=256, count=16, tri_max=60000),
        # optimising a large grid from several views
        dict(name="adjoint_256", kind="adjoint", W=512, H=512, res=256, views=8, cones32=False, grad=True),
        # the same at the size of a quick experiment
        dict(name="adjoint_32", kind="adjoint", W=61, H=47, res=32, views=2, cones32=False, grad=True),
        # the pass after the trace, default blur
        dict(name="filter_1080p", kind="filter", W=1920, H=1080, bilateral=False, tonemap=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A window of lo..hi pixels, aspect 1:1 to 2:1, odd sizes among them."""
    n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    a = rng.uniform(1.0, 2.0)
    return max(16, int(math.sqrt(n * a))), max(16, int(math.sqrt(n / a)))


def draw(rng):
    kind = rng.choice(["frame", "frame", "moving", "baked", "dense", "dense", "svo", "batch", "adjoint", "filter"])
    if kind == "frame":
        W, H = _size(rng, 14400, 2073600)
        return dict(kind=kind, W=W, H=H, res=rng.choice([32, 64, 128]), levels=rng.randint(3, 6),
                    half=rng.random() < 0.6, cones32=rng.random() < 0.25, samples=rng.choice([1, 1, 4]),
                    shadow=_log(rng, 512, 2048), ao=rng.random() < 0.25)
    if kind == "moving":
        W, H = _size(rng, 14400, 360000)
        return dict(kind=kind, W=W, H=H, res=rng.choice([32, 64, 128]), levels=rng.randint(3, 5),
                    half=rng.random() < 0.6, shadow=_log(rng, 512, 2048))
    if kind == "baked":
        W, H = _size(rng, 14400, 240000)
        return dict(kind=kind, W=W, H=H, res=rng.choice([32, 64]), levels=rng.randint(3, 5),
                    half=rng.random() < 0.6, cones32=rng.random() < 0.25, shadow=_log(rng, 256, 1024))
    if kind == "dense":
        W, H = _size(rng, 14400, 780000)
        return dict(kind=kind, W=W, H=H, res=rng.choice([32, 64, 128, 256]), tris=_log(rng, 2100, 300000),
                    cones32=rng.random() < 0.25, samples=rng.choice([1, 1, 4]))
    if kind == "svo":
        W, H = _size(rng, 14400, 230000)
        return dict(kind=kind, W=W, H=H, level=rng.randint(5, 9), tris=_log(rng, 21260, 900000),
                    shadow=_log(rng, 512, 2048))
    if kind == "batch":
        W, H = _size(rng, 14400, 65000)
        return dict(kind=kind, W=W, H=H, count=rng.randint(4, 16), tri_max=_log(rng, 10000, 60000))
    if kind == "adjoint":
        W, H = _size(rng, 2000, 66000)
        return dict(kind=kind, W=W, H=H, res=rng.choice([16, 32, 64, 128]), views=rng.randint(1, 4),
                    cones32=rng.random() < 0.25, grad=rng.random() < 0.8)
    W, H = _size(rng, 14400, 2073600)
    return dict(kind=kind, W=W, H=H, bilateral=rng.random() < 0.5, tonemap=rng.random() < 0.5)


# ---------------------------------------------------------------- device views
class _DeviceArray:
    """Device memory of the library as torch sees it; keeps its owner alive."""

    def __init__(self, ptr, words, owner):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=(int(words),), typestr="<i4", data=(int(ptr), False), version=3,
                                             strides=None)


def _words(ptr, words, owner):
    return torch.as_tensor(_DeviceArray(ptr, words, owner), device="cuda")


class _Handle:
    """A vct_dense or vct_batch handle destroyed with its last user."""

    def __init__(self, create, destroy, *args):
        self.h, self._destroy = C.c_void_p(), destroy
        A.call(create, C.byref(self.h), *args)

    def __del__(self):
        if self.h:
            A.call(self._destroy, self.h)


def _stream():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


# ---------------------------------------------------------------- clipmap frames
def _shadow_map(ctx, ds, ls, n):
    depth = torch.empty((n, n), dtype=torch.float32, device="cuda")
    A.call("vct_raycast_shadow", ctx._h, _stream(), C.byref(ds.mesh), C.byref(ls), C.c_void_p(depth.data_ptr()), n, n)
    return depth


def _rough(g, seed):
    """Per-pixel perceptual roughness U[0.1, 0.8] in the diffuse alpha byte."""
    r = torch.rand(g["depth"].shape, generator=_gen(seed), device="cuda") * 0.7 + 0.1
    g["diffuse"] = (g["diffuse"] & 0x00FFFFFF) | (torch.round(r * 255.0).to(torch.int32) << 24)
    return g


def _clipmap(case, seed):
    """Scene, context, light and G-buffer of a clipmap program."""
    scene = scenes.room(seed, scale=SCALE)
    ds = V.DeviceScene(scene)
    quirks = A.QUIRK_ALL & ~QUIRK_CLAMP_X_RANGE if case["kind"] == "moving" else A.QUIRK_ALL
    ctx = V.Context(resolution=case["res"], levels=case["levels"],
                    radiance_format=V.FORMAT_RGBA16F if case["half"] else V.FORMAT_RGBA8, quirks=quirks,
                    raster_samples=case.get("samples", 1), downsample_region_size=min(10, case["res"] // 8),
                    extent_l0=SCALE)
    W, H = case["W"], case["H"]
    cam3 = scenes.camera(seed, W, H, scale=SCALE)
    ctx.update_clip_regions(cam3[2])
    ld, ls = V.light_structs(scenes.light(seed, scale=SCALE))
    sm = V.shadow_struct(_shadow_map(ctx, ds, ls, case["shadow"]))
    gb = V.gbuffer_struct(_rough(workloads.gbuffer(ctx._h, ds, scene, cam3, W, H), seed))
    return ds, ctx, ld, ls, sm, gb, V.camera_ubo(*cam3), cam3


def _image(case):
    return torch.zeros((case["H"], case["W"], 4), dtype=torch.float32, device="cuda")


def _prepare_frame(case, seed):
    ds, ctx, ld, ls, sm, gb, cam, _ = _clipmap(case, seed)
    d, s = _image(case), _image(case)
    mgr = passes.RenderPassManager()
    mgr.add_render_pass("VoxelizationPass", passes.VoxelizationPass(ctx, ds))
    inj = passes.RadianceInjectionPass(ctx, ds, sm, ld, ls)
    mgr.add_render_pass("RadianceInjectionPass", inj)
    trace = passes.VoxelConeTracingPass(ctx, gb, cam, sm, ld, ls, d, s,
                                        A.MODE_AMBIENT_OCCLUSION if case["ao"] else A.MODE_COMBINED_GI)
    trace.enable_32_cones = case["cones32"]
    mgr.add_render_pass("VoxelConeTracingPass", trace)
    return dict(mgr=mgr, inj=inj, d=d, s=s, ao=case["ao"], ctx=ctx)


def _draw(mgr, frame, names=("VoxelizationPass", "RadianceInjectionPass", "VoxelConeTracingPass")):
    for name in names:
        mgr.draw_single_render_pass(name, frame)


def _run_frame(st):
    st["inj"].frame_index = 0  # every clip level is due
    _draw(st["mgr"], V.Frame())
    return [st["d"]] if st["ao"] else [st["d"], st["s"]]


def _prepare_moving(case, seed):
    ds, ctx, ld, ls, sm, gb, cam, cam3 = _clipmap(case, seed)
    outs = [(_image(case), _image(case)) for _ in range(MOVING_FRAMES)]
    mgr = passes.RenderPassManager()
    vox = passes.VoxelizationPass(ctx, ds, incremental=True)
    inj = passes.RadianceInjectionPass(ctx, ds, sm, ld, ls)
    trace = passes.VoxelConeTracingPass(ctx, gb, cam, sm, ld, ls, *outs[0])
    mgr.add_render_pass("VoxelizationPass", vox)
    mgr.add_render_pass("RadianceInjectionPass", inj)
    mgr.add_render_pass("VoxelConeTracingPass", trace)
    # a round trip of a few level-0 voxels a frame, ending where it began
    vs = SCALE / case["res"]
    r = np.random.default_rng(seed)
    d = vs * r.uniform(2.2, 5.0, 3) * r.choice([-1.0, 1.0], 3)
    eye = np.asarray(cam3[2], np.float64)
    path = [eye + d * k for k in ((1, 0, 0), (1, 1, 0), (1, 1, 1), (0, 0, 0))]
    vox.camera_pos = path[-1]
    _draw(mgr, V.Frame(), ("VoxelizationPass",))  # the program's first frame has voxelized every level
    return dict(mgr=mgr, vox=vox, inj=inj, trace=trace, outs=outs, path=path, ctx=ctx)


def _run_moving(st):
    st["inj"].frame_index = 0
    for k, (d, s) in enumerate(st["outs"]):
        st["vox"].camera_pos = st["path"][k]
        st["trace"].diffuse_out, st["trace"].specular_out = d, s
        _draw(st["mgr"], V.Frame(frame_index=k))
    return [im for pair in st["outs"] for im in pair]


# ---------------------------------------------------------------- analytic room
def _spheres(seed, scale):
    r = np.random.default_rng(seed + 77)
    rad = r.uniform(0.05, 0.14, 12)
    c = r.uniform(0.15, 0.85, (12, 3))
    t = lambda v: torch.tensor(v * scale, dtype=torch.float64, device="cuda")  # noqa: E731
    return t(c), t(rad)


def _view(seed, W, H, scale, obj=0):
    """G-buffer of the analytic room (the cube [0, scale]^3 seen from inside,
    with spheres), its camera triple."""
    cam3 = scenes.camera(seed, W, H, scale=scale)
    vp, vpi, eye = (torch.tensor(np.asarray(x, np.float64), device="cuda") for x in cam3)
    y, x = torch.meshgrid(torch.arange(H, device="cuda", dtype=torch.float64),
                          torch.arange(W, device="cuda", dtype=torch.float64), indexing="ij")
    q = torch.stack([(x + 0.5) / W * 2 - 1, (y + 0.5) / H * 2 - 1, torch.full_like(x, 0.5), torch.ones_like(x)], -1)
    p = q @ vpi.T
    d = p[..., :3] / p[..., 3:] - eye
    d = d / d.norm(dim=-1, keepdim=True)
    wall = torch.where(d > 0, (scale - eye) / d, -eye / d)
    wall = torch.where(d.abs() < 1e-12, torch.full_like(wall, 1e30), wall)
    t, axis = wall.min(-1)
    n = torch.zeros_like(d).scatter_(-1, axis[..., None], -torch.sign(d.gather(-1, axis[..., None])))
    mat = axis + 3 * (d.gather(-1, axis[..., None])[..., 0] > 0)
    cen, rad = _spheres(obj, scale)
    for k in range(len(rad)):
        o = eye - cen[k]
        b = (d * o).sum(-1)
        disc = b * b - (o @ o) + rad[k] ** 2
        ts = -b - torch.sqrt(disc.clamp_min(0))
        hit = (disc > 0) & (ts > 1e-3) & (ts < t)
        t = torch.where(hit, ts, t)
        n = torch.where(hit[..., None], (o + d * ts[..., None]) / rad[k], n)
        mat = torch.where(hit, torch.full_like(mat, 6 + k), mat)
    p = eye + d * t[..., None]
    c = torch.cat([p, torch.ones_like(p[..., :1])], -1) @ vp.T
    depth = (c[..., 2] / c[..., 3]).to(torch.float32)
    g = _gen(seed)
    col = torch.rand((2, 18, 4), generator=g, device="cuda") * 0.6 + 0.2
    pack = lambda v: (torch.round(v * 255).to(torch.int32) << torch.tensor([0, 8, 16, 24], device="cuda",  # noqa: E731
                                                                           dtype=torch.int32)).sum(-1).to(torch.int32)
    nrm = torch.cat([n * 0.5 + 0.5, torch.ones_like(n[..., :1])], -1).to(torch.float16).view(torch.int16)
    gb = dict(diffuse=pack(col[0])[mat], specular=pack(col[1])[mat], normal=nrm.contiguous(),
              emission=torch.zeros((H, W, 4), dtype=torch.int16, device="cuda"), depth=depth.contiguous())
    return _rough(gb, seed), cam3


def _baked_regions(case, eye):
    """Clip regions around the eye on even cells, as the reference snaps them."""
    out = []
    for lv in range(case["levels"]):
        vs = SCALE * 2 ** lv / case["res"]
        mn = tuple(int(math.floor(float(e) / (2 * vs))) * 2 - case["res"] // 2 for e in eye)
        out.append((mn, (case["res"],) * 3, vs))
    return out


def _baked_volume(case, seed, regions):
    """[levels, 6, D, D, D, 4] float32 texels: shells of the analytic room's
    surfaces, opaque where the surface passes, coloured smoothly, the toroidal
    addressing and border of the clipmap applied."""
    res = case["res"]
    cen, rad = _spheres(seed, SCALE)
    g = _gen(seed + 1)
    freq = torch.rand((4, 3), generator=g, device="cuda") * 0.6 + 0.2
    gain = torch.rand((6, 1, 1, 1, 1), generator=g, device="cuda") * 0.6 + 0.3
    vols = []
    for mn, _, vs in regions:
        ax = []
        for k in range(3):  # the cell that texel i of this axis holds
            i = torch.arange(res, device="cuda")
            ax.append((mn[k] + torch.remainder(i - mn[k], res)).double() * vs + 0.5 * vs)
        z, y, x = torch.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
        sd = torch.minimum(torch.minimum(x, SCALE - x).abs(), torch.minimum(y, SCALE - y).abs())
        sd = torch.minimum(sd, torch.minimum(z, SCALE - z).abs())
        lo, hi = torch.minimum(x, torch.minimum(y, z)), torch.maximum(x, torch.maximum(y, z))
        sd = torch.where((lo < -vs) | (hi > SCALE + vs), torch.full_like(sd, 1e9), sd)
        for k in range(len(rad)):
            r = torch.sqrt((x - cen[k, 0]) ** 2 + (y - cen[k, 1]) ** 2 + (z - cen[k, 2]) ** 2)
            sd = torch.minimum(sd, (r - rad[k]).abs())
        a = (1.25 - sd / vs).clamp(0, 1).float()
        p = torch.stack([x, y, z], -1).float()
        col = 0.5 + 0.5 * torch.sin(p @ freq.T)
        col[..., 3] = 1.0
        t = (col * a[..., None])[None].repeat(6, 1, 1, 1, 1)
        t[..., :3] *= gain
        vols.append(torch.stack([_wrap(t[f]) for f in range(6)]))
    v = torch.stack(vols)
    return v.half().float() if case["half"] else torch.round(v * 255) / 255


def _wrap(t):
    for d in range(3):
        t = torch.cat([t.narrow(d, t.shape[d] - 1, 1), t, t.narrow(d, 0, 1)], d)
    return t


def _baked_shadow(case, seed):
    n = case["shadow"]
    g = _gen(seed + 2)
    low = torch.rand((1, 1, 8, 8), generator=g, device="cuda") * 0.6 + 0.2
    return torch.nn.functional.interpolate(low, size=(n, n), mode="bilinear", align_corners=True)[0, 0].contiguous()


def _baked_desc(case, regions):
    vs = regions[0][2]
    center = [(m + case["res"] * 0.5) * vs for m in regions[0][0]]
    return A.ConeTracingDesc(A.f3(*center), A.MODE_COMBINED_GI, vs, float(case["res"]), 1.0, 8.0, 0.5, 1.0, 3.0, 2.0,
                             int(case["cones32"]))


def _prepare_baked(case, seed):
    g, cam3 = _view(seed, case["W"], case["H"], SCALE, seed)
    regions = _baked_regions(case, cam3[2])
    ctx = V.Context(resolution=case["res"], levels=case["levels"],
                    radiance_format=V.FORMAT_RGBA16F if case["half"] else V.FORMAT_RGBA8,
                    downsample_region_size=min(10, case["res"] // 8), extent_l0=SCALE)
    ctx.set_regions(regions)
    v = _baked_volume(case, seed, regions)  # L, F, z, y, x, 4 -> the atlas z, (L y), (F x), 4
    v = v.permute(2, 0, 3, 1, 4, 5).contiguous()
    if case["half"]:
        host = v.half().view(torch.int16).cpu().numpy().view(np.uint16)
    else:
        host = torch.round(v * 255).to(torch.uint8).cpu().numpy().view(np.uint32)
    ctx.write_volume(V.VOLUME_RADIANCE, host)
    ld, ls = V.light_structs(scenes.light(seed, scale=SCALE))
    return dict(ctx=ctx, gb=V.gbuffer_struct(g), cam=V.camera_ubo(*cam3), desc=_baked_desc(case, regions), ld=ld, ls=ls,
                sm=V.shadow_struct(_baked_shadow(case, seed)), d=_image(case), s=_image(case))


def _run_baked(st):
    st["ctx"].trace(st["gb"], st["cam"], st["desc"], st["sm"], st["ld"], st["ls"], st["d"], st["s"])
    return [st["d"], st["s"]]


# ---------------------------------------------------------------- dense method
def _thin_room(seed, tris):
    """The room with as many of its 16 spheres as `tris` holds, topped up with thin triangles."""
    return scenes.room(seed, n_spheres=int(min(16, max(0, (tris - 780) // 1280))), thin_total=tris)


def _trace_desc(case):
    td = workloads.dense_trace_desc(math.sqrt(3.0))
    td.enable_32_cones = int(case.get("cones32", False))
    td.aperture = 0.628319 if case.get("cones32", False) else 0.872665
    return td


def _prepare_dense(case, seed):
    scene = _thin_room(seed, case["tris"])
    ds = V.DeviceScene(scene)
    W, H = case["W"], case["H"]
    cam3 = scenes.camera(seed, W, H)
    sc = workloads.scratch_ctx()
    g = workloads.gbuffer(sc, ds, scene, cam3, W, H)
    A.call("vct_destroy", sc)
    gmin, ext = workloads.grid_box(scene)
    grid = _Handle("vct_dense_create", "vct_dense_destroy",
                   C.byref(A.DenseDesc(A.f3(*gmin), ext, case["res"], 0, case["samples"], 0)))
    p, b, f = C.c_void_p(), C.c_size_t(), C.c_uint32()
    total, first = 0, None
    for m in range(case["res"].bit_length()):
        A.call("vct_dense_level", grid.h, m, C.byref(p), C.byref(b), C.byref(f))
        first = p.value if first is None else first
        total = p.value + b.value - first
    return dict(ds=ds, gb=V.gbuffer_struct(g), cam=V.camera_ubo(*cam3), td=_trace_desc(case), grid=grid, out=_image(case),
                pyramid=_words(first, total // 4, grid))


def _run_dense(st):
    s, h = _stream(), st["grid"].h
    A.call("vct_dense_clear", h, s)
    A.call("vct_dense_voxelize", h, s, C.byref(st["ds"].mesh))
    A.call("vct_dense_mipmap", h, s)
    A.call("vct_dense_trace", h, s, C.byref(st["gb"]), C.byref(st["cam"]), C.byref(st["td"]),
           C.c_void_p(st["out"].data_ptr()), None)
    return [st["out"], st["pyramid"]]


# ---------------------------------------------------------------- octree
def _prepare_svo(case, seed):
    scene = scenes.room(seed, thin_total=case["tris"])
    ds = V.DeviceScene(scene)
    ctx = V.Context(resolution=16, levels=1, downsample_region_size=1, extent_l0=1.0)
    ld, ls = V.light_structs(scenes.light(seed))
    sm = V.shadow_struct(_shadow_map(ctx, ds, ls, case["shadow"]))
    W, H = case["W"], case["H"]
    cam3 = scenes.camera(seed, W, H)
    gb = V.gbuffer_struct(workloads.gbuffer(ctx._h, ds, scene, cam3, W, H))
    dim = 1 << case["level"]
    desc = A.ConeTracingDesc(A.f3(0.5, 0.5, 0.5), A.MODE_COMBINED_GI, 1.0 / dim, float(dim), 1.0, 8.0, 0.5, 1.0, 3.0,
                             2.0, 0)
    return dict(ds=ds, ctx=ctx, ld=ld, ls=ls, sm=sm, gb=gb, cam=V.camera_ubo(*cam3), level=case["level"], desc=desc,
                lo=(C.c_float * 3)(*scene.bb_min.tolist()), hi=(C.c_float * 3)(*scene.bb_max.tolist()),
                d=_image(case), s=_image(case),
                # the program's own copy of the node pool, with room for any seed's
                nodes=torch.zeros(2 * min(8 * dim ** 3, 16 << 20), dtype=torch.int32, device="cuda"))


def _run_svo(st):
    s, h, n, pool = _stream(), st["ctx"]._h, C.c_uint32(), C.c_void_p()
    A.call("vct_svo_voxelize", h, s, C.byref(st["ds"].mesh), C.byref(st["sm"]), C.byref(st["ld"]), C.byref(st["ls"]),
           st["level"], C.byref(n))
    A.call("vct_svo_build", h, s)
    A.call("vct_svo_trace", h, s, C.byref(st["gb"]), C.byref(st["cam"]), C.byref(st["desc"]), C.byref(st["sm"]),
           C.byref(st["ld"]), C.byref(st["ls"]), st["lo"], st["hi"], C.c_void_p(st["d"].data_ptr()),
           C.c_void_p(st["s"].data_ptr()), None)
    nodes = C.c_uint32()
    A.call("vct_svo_pool", h, C.byref(pool), C.byref(nodes))
    k = min(2 * nodes.value, st["nodes"].numel())
    st["nodes"][:k].copy_(_words(pool.value, k, st["ctx"]))
    return [st["d"], st["s"], int(n.value), st["nodes"]]


# ---------------------------------------------------------------- batch
def _prepare_batch(case, seed):
    items = []
    sc = workloads.scratch_ctx()
    W, H = case["W"], case["H"]
    for i, (tris, res) in enumerate(scenes.batch_sizes(seed, case["count"], 5000, case["tri_max"])):
        scene = _thin_room(seed + i, tris)
        ds = V.DeviceScene(scene)
        cam3 = scenes.camera(seed + i, W, H)
        gmin, ext = workloads.grid_box(scene)
        items.append(dict(ds=ds, res=res, gb=V.gbuffer_struct(workloads.gbuffer(sc, ds, scene, cam3, W, H)),
                          cam=V.camera_ubo(*cam3), gmin=gmin, ext=ext, out=_image(case)))
    A.call("vct_destroy", sc)
    td = _trace_desc(case)
    b = _Handle("vct_batch_create", "vct_batch_destroy", workloads.batch_scene_array(items), len(items), C.byref(td))
    return dict(batch=b, items=items)


def _run_batch(st):
    A.call("vct_batch_run", st["batch"].h, _stream(), None)
    return [it["out"] for it in st["items"]]


# ---------------------------------------------------------------- adjoint
def _adjoint_params(case):
    from vk_voxel_cone_tracing_amd import adjoint as adj

    return adj.TraceParams(aperture=0.628319 if case["cones32"] else 0.872665, max_distance=math.sqrt(3.0),
                           enable_32_cones=int(case["cones32"]))


def _prepare_adjoint(case, seed):
    from vk_voxel_cone_tracing_amd import adjoint as adj

    n, W, H = case["views"], case["W"], case["H"]
    gs, cams = zip(*[_view(seed + v, W, H, 1.0, seed) for v in range(n)])
    st = {k: torch.stack([g[k] for g in gs]).contiguous() for k in ("diffuse", "normal", "depth")}
    gen, r = _gen(seed), case["res"]
    albedo = torch.rand((r, r, r, 3), generator=gen, device="cuda") * 0.6 + 0.2
    opacity = torch.rand((r, r, r), generator=gen, device="cuda") * 0.5 + 0.05
    target = torch.rand((n, H, W, 4), generator=gen, device="cuda")
    return dict(st, cameras=adj.cameras_tensor(cams), albedo=albedo.requires_grad_(case["grad"]),
                opacity=opacity.requires_grad_(case["grad"]), target=target, p=_adjoint_params(case), adj=adj)


def _run_adjoint(st):
    a, o = st["albedo"], st["opacity"]
    out = st["adj"].render(a, o, st["diffuse"], st["normal"], st["depth"], st["cameras"], (0.0, 0.0, 0.0), 1.0, st["p"])
    if not a.requires_grad:
        return [out]
    a.grad = o.grad = None
    ((out - st["target"]) ** 2).sum().backward()
    return [out.detach(), a.grad, o.grad]


# ---------------------------------------------------------------- filter
def _prepare_filter(case, seed):
    """A traced frame's two images: smooth shading with object edges, the
    specular one noisy from pixel to pixel (roughness varies)."""
    H, W, g = case["H"], case["W"], _gen(seed)
    up = lambda k: torch.nn.functional.interpolate(torch.rand((1, 4, k, k), generator=g, device="cuda"),  # noqa: E731
                                                   size=(H, W), mode="nearest")[0].permute(1, 2, 0)
    d = (up(9) * 2 + 0.2 * torch.rand((H, W, 4), generator=g, device="cuda")).contiguous()
    s = (up(13) * (0.5 + torch.rand((H, W, 4), generator=g, device="cuda"))).contiguous()
    return dict(d=d, s=s, out=_image(case), W=W, H=H,
                desc=A.SpecularFilterDesc(2.2, 0.1, int(case["tonemap"]), 0 if case["bilateral"] else 1))


def _run_filter(st):
    A.call("vct_specular_filter", _stream(), C.c_void_p(st["d"].data_ptr()), C.c_void_p(st["s"].data_ptr()), st["W"],
           st["H"], C.byref(st["desc"]), C.c_void_p(st["out"].data_ptr()))
    return st["out"]


def prepare(case, seed):
    return dict(globals()["_prepare_" + case["kind"]](case, int(seed) % 1000003), kind=case["kind"])


def run(state):
    return globals()["_run_" + state["kind"]](state)


# ---------------------------------------------------------------- work
def _cone_steps(aperture, vs, reach, factor=1.0):
    """Steps of one cone march: voxel-sized until the cone is wider, then geometric."""
    coef, t, n = 2 * math.tan(aperture / 2), 0.0, 0
    while t < reach and n < 4000:
        t += max(t * coef, vs) * factor
        n += 1
    return n


def work(case):
    """Inputs read once, outputs written once; the trilinear filtering of the
    cone samples of half the cones (the hemisphere above a surface)."""
    k, px = case["kind"], case["W"] * case["H"]
    if k in ("frame", "moving", "baked"):
        D = case["res"] + 2
        texels = case["levels"] * 6 * D ** 3
        vs = SCALE / case["res"]
        cones = 16 if case.get("cones32") else 8
        steps = cones * _cone_steps(0.628319 if case.get("cones32") else 0.872665, vs, 30.0)
        if not case.get("ao"):
            steps += _cone_steps(0.45, vs, 30.0, vs)
        tb = 8 if case["half"] else 4
        image = px * (28 + 32) + 4 * case["shadow"] ** 2
        flops = px * steps * 384
        if k == "baked":
            return {"bytes": texels * tb + image, "flops": flops}
        frame = texels * (4 + tb) + texels * tb + image + 21260 * 100
        if k == "frame":
            return {"bytes": frame, "flops": flops}
        return {"bytes": MOVING_FRAMES * (texels * tb + image), "flops": MOVING_FRAMES * flops}
    if k == "dense":
        n = case["res"]
        texels = n ** 3 * (1 + 6 / 7)
        steps = (16 if case["cones32"] else 8) * _cone_steps(0.628319 if case["cones32"] else 0.872665, 1 / n, 1.732)
        return {"bytes": texels * 4 * 2 + px * (16 + 16) + case["tris"] * 100, "flops": px * steps * 384}
    if k == "svo":
        n = 1 << case["level"]
        frags = 6 * n * n + 5 * case["tris"]
        steps = 8 * _cone_steps(0.872665, 1 / n, 1.732)
        return {"bytes": frags * 16 + frags * 2 * 8 * 2 + px * 60 + case["tris"] * 100, "flops": px * steps * 40}
    if k == "batch":
        c, n = case["count"], 128
        steps = 8 * _cone_steps(0.872665, 1 / n, 1.732)
        return {"bytes": c * (n ** 3 * 4 * 2 + px * 32 + 20000 * 100), "flops": c * px * steps * 384}
    if k == "adjoint":
        n, v = case["res"], case["views"]
        steps = (16 if case["cones32"] else 8) * _cone_steps(0.628319 if case["cones32"] else 0.872665, 1 / n, 1.732)
        f = 3 if case["grad"] else 1
        return {"bytes": f * n ** 3 * 16 + v * px * (16 + 16 * f), "flops": f * v * px * steps * 384}
    return {"bytes": px * 48, "flops": px * (225 * 12 if case["bilateral"] else 9 * 8)}


def tolerance(case):
    """About four times the difference between this code and a build of it
    without contracted multiply-adds, over the listed and drawn cases (largest
    seen, rel / max: clipmap frames 2e-5 / 8e-3, baked 1e-4 / 4e-3, dense
    3e-4 / 0.5 at one pixel of one view, batch 1.3e-4 / 2e-3, octree 2e-6 /
    8e-4, adjoint 5e-5 / 2e-3); the filter, whose sums are never contracted,
    is within 8e-7 of float64. Octree pools, fragment counts and the bytes of
    dense pyramids are whole numbers and do not differ at all."""
    return {"frame": {"rel": 1e-4, "max": 0.03}, "moving": {"rel": 1e-4, "max": 0.03},
            "baked": {"rel": 4e-4, "max": 0.02}, "dense": {"rel": 1e-3, "max": 0.95},
            "batch": {"rel": 5e-4, "max": 0.02}, "svo": {"rel": 2e-5, "max": 0.01},
            "adjoint": {"rel": 2e-4, "max": 0.01}, "filter": {"rel": 5e-6, "max": 2e-4}}[case["kind"]]


# ---------------------------------------------------------------- float64 references
DIRS16 = [(0.57735, 0.57735, 0.57735), (0.57735, -0.57735, -0.57735), (-0.57735, 0.57735, -0.57735),
          (-0.57735, -0.57735, 0.57735), (-0.903007, -0.182696, -0.388844), (-0.903007, 0.182696, 0.388844),
          (0.903007, -0.182696, 0.388844), (0.903007, 0.182696, -0.388844), (-0.388844, -0.903007, -0.182696),
          (0.388844, -0.903007, 0.182696), (0.388844, 0.903007, -0.182696), (-0.388844, 0.903007, 0.182696),
          (-0.182696, -0.388844, -0.903007), (0.182696, 0.388844, -0.903007), (-0.182696, 0.388844, 0.903007),
          (0.182696, -0.388844, 0.903007)]


def _dirs32():
    a, b, c, e = 0.898904, 0.435512, 0.0479745, 0.57735
    base = [(a, b, c), (a, -b, -c), (a, c, -b), (a, -c, b), (-a, b, -c), (-a, -b, c), (-a, c, b), (-a, -c, -b),
            (c, a, b), (-c, a, -b), (-b, a, c), (b, a, -c), (-c, -a, b), (c, -a, -b), (b, -a, c), (-b, -a, -c),
            (b, c, a), (-b, -c, a), (c, -b, a), (-c, b, a), (b, -c, -a), (-b, c, -a), (c, b, -a), (-c, -b, -a)]
    return base + [(x * e, y * e, z * e) for x in (1, -1) for y in (1, -1) for z in (1, -1)]


def _f64(x):
    return torch.as_tensor(x, device="cuda").double()


def _bytes4(t):
    return torch.stack([(t >> s) & 255 for s in (0, 8, 16, 24)], -1).double() / 255


def _surface(g, cam3, W, H, idx):
    """World position, unit normal and view of the pixels `idx` (flat)."""
    vpi = _f64(np.asarray(cam3[1], np.float32))
    eye = _f64(np.asarray(cam3[2], np.float32))
    depth = g["depth"].reshape(-1)[idx].double()
    q = torch.stack([((idx % W).double() + 0.5) / W * 2 - 1, ((idx // W).double() + 0.5) / H * 2 - 1, depth,
                     torch.ones_like(depth)], -1)
    p = q @ vpi.T
    world = p[:, :3] / p[:, 3:]
    n = g["normal"].reshape(-1, 4)[idx].view(torch.float16)[:, :3].double() * 2 - 1
    n = n / n.norm(dim=-1, keepdim=True)
    view = eye - world
    return world, n, view / view.norm(dim=-1, keepdim=True)


def _corners(u, top):
    """Corner index and weight of the 8 texels around u (..., 3), index clamped to [0, top]."""
    f = torch.floor(u)
    w = u - f
    for c in range(8):
        o = torch.tensor([c & 1, (c >> 1) & 1, c >> 2], device=u.device)
        i = (f.long() + o).clamp(min=0)
        i = torch.minimum(i, top)
        ww = torch.where(o.bool(), w, 1 - w).prod(-1)
        yield i, ww


def _clip_sample(vol, case, vs, pos, level, face, wts):
    """vol: [L * 6 * D^3, 4] float64; level (n,) long; face (n, 3), wts (n, 3)."""
    D, res = case["res"] + 2, case["res"]
    ext = vs * res * torch.pow(2.0, level.double())
    q = pos / ext[:, None]
    u = (q - torch.floor(q)) * res + 0.5
    out = torch.zeros((len(pos), 4), dtype=torch.float64, device="cuda")
    top = torch.tensor(D - 1, device="cuda")
    for i, w in _corners(u, top):
        cell = (i[:, 2] * D + i[:, 1]) * D + i[:, 0]
        for a in range(3):
            out += vol[(level * 6 + face[:, a]) * D ** 3 + cell] * (w * wts[:, a])[:, None]
    return out


def _clip_cone(vol, case, center, vs, start, d, aperture, start_level, factor):
    """Front-to-back march of one cone per row; returns rgb and 1 - occlusion."""
    n, L = len(start), case["levels"]
    coef = 2 * torch.tan(aperture / 2)
    vs0 = vs * torch.pow(2.0, start_level)
    pos0 = start + d * (vs0 * 0.5)[:, None]
    face = torch.tensor([0, 2, 4], device="cuda") + (d <= 0).long()
    wts = d * d
    rmin = vs * case["res"] * 0.5
    rgb = torch.zeros((n, 3), dtype=torch.float64, device="cuda")
    occ_out = torch.zeros(n, dtype=torch.float64, device="cuda")
    act = torch.arange(n, device="cuda")
    step = torch.zeros(n, dtype=torch.float64, device="cuda")
    alpha, occ, seg = torch.zeros_like(step), torch.zeros_like(step), vs0.clone()
    diam = torch.full_like(step, vs)
    while len(act):
        pos = pos0 + d * step[:, None]
        dist = (center - pos).norm(dim=-1)
        cur = torch.maximum(torch.maximum(start_level, torch.log2(diam / vs)), torch.ceil(torch.log2(dist / rmin)))
        cur = cur.clamp(max=L - 1)
        lo = torch.floor(cur)
        fl = (cur - lo)[:, None]
        s = _clip_sample(vol, case, vs, pos, lo.long(), face, wts) * (1 - fl)
        s = s + _clip_sample(vol, case, vs, pos, torch.ceil(cur).long(), face, wts) * fl
        vsl = vs * torch.pow(2.0, cur)
        corr = seg / vsl
        op = (1 - torch.pow((1 - s[:, 3]).clamp(min=0), corr)).clamp(0, 1)
        blend = (1 - alpha).clamp(0, 1)
        rgb[act] += blend[:, None] * s[:, :3] * corr[:, None]
        alpha = alpha + blend * op
        occ = occ + (1 - occ) * op / (1 + (step + vsl) * 2.0)
        nxt = step + diam.clamp(min=vs) * factor
        seg, step = nxt - step, nxt
        diam = step * coef
        occ_out[act] = occ
        keep = (step < 30.0) & (occ < 1.0)
        if not bool(keep.all()):
            act, step, alpha, occ, seg, diam = (t[keep] for t in (act, step, alpha, occ, seg, diam))
            pos0, d, face, wts, start_level, coef = (t[keep] for t in (pos0, d, face, wts, start_level, coef))
    return rgb, 1 - occ_out


def _brdf(n, v, l, dc, sc, rough):
    dot = lambda a, b: (a * b).sum(-1)  # noqa: E731
    pi, al = 3.141592, rough * rough
    r90 = (sc.max(-1).values * 50).clamp(0, 1)
    h = l + v
    h = h / h.norm(dim=-1, keepdim=True)
    ndl, ndv = dot(n, l).clamp(0.001, 1), dot(n, v).abs().clamp(0.001, 1)
    ndh, vdh = dot(n, h).clamp(0, 1), dot(v, h).clamp(0, 1)
    att = lambda x: 2 * x / (x + torch.sqrt(al * al + (1 - al * al) * x * x))  # noqa: E731
    f = (ndh * al * al - ndh) * ndh + 1
    dd = al * al / (pi * f * f)
    fres = sc + (r90[:, None] - sc) * ((1 - vdh).clamp(0, 1) ** 5)[:, None]
    spec = fres * (att(ndl) * att(ndv) * dd / (4 * ndl * ndv))[:, None]
    return ndl[:, None] * ((1 - fres) * dc / pi + spec)


def _pcf(depth, light, world):
    """16 bilinear taps of raw light depth around the projected point, zero outside the map."""
    h, w = depth.shape
    view, proj = _f64(np.asarray(light["view"], np.float32)), _f64(np.asarray(light["proj"], np.float32))
    p = torch.cat([world, torch.ones_like(world[:, :1])], -1) @ view.T
    xy = p[:, :2] * torch.stack([proj[0, 0], proj[1, 1]]) + proj[:2, 3] + p[:, [1, 0]] * torch.stack(
        [proj[0, 1], proj[1, 0]])
    xy = xy * 0.5 + 0.5
    d = torch.nn.functional.pad(depth.double(), (1, 1, 1, 1))
    out = torch.zeros(len(world), dtype=torch.float64, device="cuda")
    for yi in range(4):
        for xi in range(4):
            u, v = xy[:, 0] * w + (xi - 1.5) - 0.5, xy[:, 1] * h + (yi - 1.5) - 0.5
            fu, fv = torch.floor(u), torch.floor(v)
            a, b = u - fu, v - fv
            i, j = fu.clamp(-4, w + 4).long(), fv.clamp(-4, h + 4).long()
            tap = lambda x, y: d[(y + 1).clamp(0, h + 1), (x + 1).clamp(0, w + 1)]  # noqa: E731
            out += ((1 - a) * (1 - b) * tap(i, j) + a * (1 - b) * tap(i + 1, j) + (1 - a) * b * tap(i, j + 1)
                    + a * b * tap(i + 1, j + 1))
    return out / 16


def _exact_baked(case, seed):
    W, H = case["W"], case["H"]
    g, cam3 = _view(seed, W, H, SCALE, seed)
    regions = _baked_regions(case, cam3[2])
    vol = _baked_volume(case, seed, regions).double().reshape(-1, 4)
    desc = _baked_desc(case, regions)
    center, vs = _f64(list(desc.volume_center)), regions[0][2]
    light = scenes.light(seed, scale=SCALE)
    ldir = -_f64(np.asarray(light["direction"], np.float32))
    ldir = ldir / ldir.norm()
    shadow = _baked_shadow(case, seed)
    dirs = _f64(np.asarray(_dirs32() if case["cones32"] else DIRS16, np.float32))
    ap = torch.tensor(float(np.float32(0.628319 if case["cones32"] else 0.872665)), dtype=torch.float64, device="cuda")
    rmin = vs * case["res"] * 0.5
    out_d = torch.zeros((H * W, 4), dtype=torch.float64, device="cuda")
    out_s = torch.zeros_like(out_d)
    out_d[:, 3] = out_s[:, 3] = 1
    for idx in torch.arange(H * W, device="cuda").split(40000):
        world, n, view = _surface(g, cam3, W, H, idx)
        dif, spec = _bytes4(g["diffuse"].reshape(-1)[idx]), _bytes4(g["specular"].reshape(-1)[idx])
        dist = (center - world).norm(dim=-1)
        ml = torch.log2(dist / rmin).clamp(min=0)
        f = dist / (rmin * torch.pow(2.0, torch.ceil(ml)))
        start_level = torch.where(f > 0.5, torch.ceil(ml) + (f - 0.5) * 2, torch.ceil(ml))
        start = world + n * (vs * torch.pow(2.0, start_level))[:, None]
        ind = torch.zeros((len(idx), 4), dtype=torch.float64, device="cuda")
        ind[:, 3] = 1
        for k in range(len(dirs)):
            ct = n @ dirs[k]
            m = ct >= 0
            if not bool(m.any()):
                continue
            rgb, vis = _clip_cone(vol, case, center, vs, start[m], dirs[k].expand(int(m.sum()), 3),
                                  ap.expand(int(m.sum())), start_level[m], 1.0)
            ind[m] += torch.cat([rgb, vis[:, None]], -1) * ct[m][:, None]
        ind = ind / len(dirs)
        ao = ind[:, 3] * 0.5
        direct = _brdf(n, view, ldir, dif[:, :3], spec[:, :3], dif[:, 3]) * _pcf(shadow, light, world)[:, None]
        out_d[idx, :3] = direct * ao[:, None] + ind[:, :3] * dif[:, :3] * 8.0
        refl = -view + 2 * (n * view).sum(-1, keepdim=True) * n
        m = (spec[:, :3].max(-1).values > 1e-6) & (spec[:, 3] > 1e-6)
        rgb, _ = _clip_cone(vol, case, center, vs, start[m], refl[m], dif[m][:, 3].clamp(min=0.05), start_level[m], vs)
        out_s[idx[m], :3] = rgb * spec[m][:, :3] * 3.0
    return [out_d.reshape(H, W, 4), out_s.reshape(H, W, 4)]


def _mips64(level0):
    """Level 0 [n, n, n, 4] (z, y, x) to the levels' faces, each padded by a
    zero texel: [1 or 6, D, D, D, 4]."""
    pad = lambda t: torch.nn.functional.pad(t, (0, 0, 1, 1, 1, 1, 1, 1))  # noqa: E731
    levels, faces = [pad(level0[None])], [level0] * 6
    while faces[0].shape[0] > 1:
        up = []
        for f in range(6):
            ax = 2 - (f >> 1)  # x, y, z are the last, middle and first axis
            n = faces[f].shape[0] // 2
            c = faces[f].reshape(n, 2, n, 2, n, 2, 4)
            a, b = c.select(2 * ax + 1, f & 1), c.select(2 * ax + 1, 1 - (f & 1))
            v = a + (1 - a[..., 3:]) * b
            kept = [2 * k + 1 for k in range(ax)] + [2 * k for k in range(ax + 1, 3)]
            up.append(v.mean(dim=kept))
        faces = up
        levels.append(pad(torch.stack(faces)))
    return levels


def _dense_sample(levels, m, pos, face, wts):
    """Level m (int) at pos (n, 3) in grid units [0, 1]."""
    t = levels[m]
    n = t.shape[1] - 2
    u = pos * n + 0.5  # bordered texel coordinate of texel centres
    f = torch.floor(u)
    ok = ((f >= 0) & (f <= n)).all(-1)
    top = torch.tensor(n + 1, device="cuda")
    flat = t.reshape(t.shape[0], -1, 4)
    D = n + 2
    out = torch.zeros((len(pos), 4), dtype=torch.float64, device="cuda")
    for i, w in _corners(u, top):
        cell = (i[:, 2] * D + i[:, 1]) * D + i[:, 0]
        if m == 0:
            out = out + flat[0, cell] * (w * wts.sum(-1))[:, None]
        else:
            for a in range(3):
                out = out + flat[face[:, a], cell] * (w * wts[:, a])[:, None]
    return torch.where(ok[:, None], out, torch.zeros_like(out))


def _dense_cones(levels, vs, coef, start, d):
    """The dense march of one direction for every row of start; all steps taken (no exit on full occlusion)."""
    L = len(levels)
    pos0 = start + d * (vs * 0.5)
    face = (torch.tensor([0, 2, 4], device="cuda") + (d <= 0).long()).expand(len(start), 3)
    wts = (d * d).expand(len(start), 3)
    rgb, alpha, occ = 0.0, 0.0, 0.0
    step, diam, seg = 0.0, vs, vs
    while step < float(np.float32(math.sqrt(3.0))):
        lvl = min(max(math.log2(diam / vs), 0.0), L - 1.0)
        lo, fl = int(math.floor(lvl)), lvl - math.floor(lvl)
        pos = pos0 + d * step
        s = _dense_sample(levels, lo, pos, face, wts)
        if fl > 0:
            s = s * (1 - fl) + _dense_sample(levels, lo + 1, pos, face, wts) * fl
        vsl = vs * 2 ** lvl
        corr = seg / vsl
        op = (1 - torch.pow((1 - s[:, 3]).clamp(min=1e-300), corr)).clamp(0, 1)
        blend = 1 - alpha
        rgb = rgb + (blend * corr)[:, None] * s[:, :3] if step else s[:, :3] * corr
        alpha = alpha + blend * op
        occ = occ + (1 - occ) * op / (1 + (step + vsl) * 2.0)
        nxt = step + max(diam, vs)
        seg, step = nxt - step, nxt
        diam = step * coef
    return rgb, 1 - occ


def _exact_adjoint(case, seed):
    n, W, H, r = case["views"], case["W"], case["H"], case["res"]
    if n * W * H > 100000:
        return None
    st = _prepare_adjoint(case, seed)
    a, o = st["albedo"].detach().double(), st["opacity"].detach().double()
    if case["grad"]:
        a.requires_grad_(True)
        o.requires_grad_(True)
    levels = _mips64(torch.cat([a, o[..., None]], -1))
    leaf = [t.detach().requires_grad_(case["grad"]) for t in levels]
    vs = 1.0 / r
    dirs = _f64(np.asarray(_dirs32() if case["cones32"] else DIRS16, np.float32))
    coef = 2 * math.tan(float(np.float32(st["p"].aperture)) / 2)
    out = torch.zeros((n * H * W, 4), dtype=torch.float64, device="cuda")
    for v in range(n):
        g = {k: st[k][v] for k in ("diffuse", "normal", "depth")}
        row = st["cameras"][v].numpy()
        cam3 = (None, row[16:32].reshape(4, 4).T, row[32:35])
        for idx in torch.arange(H * W, device="cuda").split(8000):
            world, nrm, _ = _surface(g, cam3, W, H, idx)
            albedo = _bytes4(g["diffuse"].reshape(-1)[idx])[:, :3]
            start = world + nrm * vs
            parts = []
            for k in range(len(dirs)):
                ct = nrm @ dirs[k]
                m = torch.nonzero(ct >= 0)[:, 0]
                if not len(m):
                    continue
                rgb, vis = _dense_cones(leaf, vs, coef, start[m], dirs[k])
                c = torch.cat([rgb, vis[:, None]], -1) * ct[m][:, None]
                parts.append(torch.zeros((len(idx), 4), dtype=torch.float64, device="cuda").index_add(0, m, c))
            ind = sum(parts) + _f64([0.0, 0.0, 0.0, 1.0])
            px = torch.cat([ind[:, :3] / len(dirs) * albedo * 8.0, ind[:, 3:] / len(dirs) * 0.5], -1)
            hit = (g["depth"].reshape(-1)[idx] != 1.0)[:, None]
            px = torch.where(hit, px, _f64([0.0, 0.0, 0.0, 1.0]).expand_as(px))
            if case["grad"]:
                t = st["target"].reshape(n, H * W, 4)[v, idx].double()
                ((px - t) ** 2).sum().backward()
            out[v * H * W + idx] = px.detach()
    out = out.reshape(n, H, W, 4)
    if not case["grad"]:
        return [out]
    torch.autograd.backward(levels, [t.grad if t.grad is not None else torch.zeros_like(t) for t in leaf])
    return [out, a.grad, o.grad]


def _tap(img, x, y):
    """Bilinear, clamped to the edge, at texel coordinates (x, y) of texel centres at integers."""
    H, W = img.shape[:2]
    fx, fy = torch.floor(x), torch.floor(y)
    a, b = (x - fx)[None, :, None], (y - fy)[:, None, None]
    i, j = fx.long(), fy.long()
    at = lambda jj, ii: img[jj.clamp(0, H - 1)][:, ii.clamp(0, W - 1)]  # noqa: E731
    return ((1 - a) * (1 - b) * at(j, i) + a * (1 - b) * at(j, i + 1) + (1 - a) * b * at(j + 1, i)
            + a * b * at(j + 1, i + 1))


def _exact_filter(case, seed):
    st = _prepare_filter(case, seed)
    d, s = st["d"].double(), st["s"].double()
    H, W = case["H"], case["W"]
    x, y = torch.arange(W, device="cuda").double(), torch.arange(H, device="cuda").double()
    col = d.clone()
    if not case["bilateral"]:
        acc = s.clone()
        a, two_pi = np.float32(0), np.float32(6.28318530718)
        while a < two_pi:  # the shader's float loop
            for i in range(1, 9):
                acc += _tap(s, x + math.cos(a) * 0.01 * i / 8, y + math.sin(a) * 0.01 * i / 8)
            a = np.float32(a + np.float32(two_pi / np.float32(32)))
        f = acc / (8.0 * 32.0 - 15.0)
        col[..., :3] += f[..., :3]
    else:
        kern = [0.031225216, 0.033322271, 0.035206333, 0.036826804, 0.038138565, 0.039104044, 0.039695028, 0.039894000]
        kern = kern + kern[-2::-1]
        z, acc = 0.0, 0.0
        for i in range(-7, 8):
            for j in range(-7, 8):
                q = _tap(s, x + i, y + j)[..., :3]
                dd = ((q - s[..., :3]) ** 2).sum(-1)
                w = torch.exp(-0.5 * dd / 100.0) * kern[7 + j] * kern[7 + i]
                z, acc = z + w, acc + w[..., None] * q
        col[..., :3] += acc / z[..., None]
    if case["tonemap"]:
        u = lambda v: (v * (0.15 * v + 0.05) + 0.004) / (v * (0.15 * v + 0.5) + 0.06) - 0.02 / 0.3  # noqa: E731
        col[..., :3] = torch.pow(u(col[..., :3] * float(np.float32(0.1))) / u(11.2), 1 / float(np.float32(2.2)))
    return col


def exact(case, seed):
    seed = int(seed) % 1000003
    if case["kind"] == "baked":
        return _exact_baked(case, seed)
    if case["kind"] == "adjoint":
        return _exact_adjoint(case, seed)
    if case["kind"] == "filter":
        return _exact_filter(case, seed)
    return None  # a whole pipeline: rasterized voxels, byte-valued mips, trace
