"""The dense mip pyramid of random level-0 texels against a NumPy float32
restatement, bit for bit, at every resolution where the launches change: the
whole pyramid in the one-workgroup tail (2 to 32, RGBA32F to 16), one or more
levels above it, and rows of 64 texels; RGBA8 and RGBA32F, and the batched
launch's bricks."""
import ctypes as C

import numpy as np
import pytest

import oracle_api as O

pytestmark = pytest.mark.gpu


def _mips(level0, fmt):
    """Faces of levels 1.. of level0 (z, y, x, 4) float32: four front-to-back
    pairs per face, listed by the child with the axis bit clear, the front
    child being that one for even faces and the other for odd ones."""
    f32 = np.float32
    faces, out = [level0] * 6, []
    while faces[0].shape[0] > 1:
        up = []
        for f in range(6):
            axis = f >> 1
            child = lambda c: faces[f][c >> 2::2, (c >> 1) & 1::2, c & 1::2]  # noqa: E731
            acc = np.zeros(child(0).shape, f32)
            for c in (c for c in range(8) if not c & (1 << axis)):
                pair = (child(c), child(c | (1 << axis)))
                a, b = pair if not f & 1 else pair[::-1]
                acc = acc + a
                acc = acc + (f32(1) - a[..., 3:]) * b
            v = acc * f32(0.25)
            if fmt == O.FMT_RGBA8:
                v = np.rint(np.clip(v, 0, 1) * f32(255)).astype(np.uint32)
                out_f, v = v, v.astype(f32) / f32(255)
            else:
                out_f = v
            up.append((out_f, v))
        faces = [v for _, v in up]
        out.append(np.stack([o for o, _ in up]))
    return out


@pytest.mark.parametrize("fmt", [O.FMT_RGBA8, O.FMT_RGBA32F])
@pytest.mark.parametrize("res", [2, 4, 16, 32, 64, 256])
def test_mips_bit_exact(res, fmt):
    import vk_voxel_cone_tracing_amd as V

    A = V._abi
    rng = np.random.default_rng(res)
    h = C.c_void_p()
    A.call("vct_dense_create", C.byref(h), C.byref(A.DenseDesc(A.f3(0, 0, 0), 1.0, res, fmt, 1, 0)))
    try:
        D = res + 2
        bytes4 = rng.integers(0, 256, (res, res, res, 4)).astype(np.uint32)
        bytes4[rng.uniform(size=bytes4.shape[:3]) < 0.4] = 0
        if fmt == O.FMT_RGBA8:
            level0 = bytes4.astype(np.float32) / np.float32(255)
            host = np.zeros((D, D, D), np.uint32)
            host[1:-1, 1:-1, 1:-1] = (bytes4 << np.arange(0, 32, 8, dtype=np.uint32)).sum(-1, dtype=np.uint32)
        else:
            level0 = rng.uniform(-0.5, 1.5, bytes4.shape).astype(np.float32)
            host = np.zeros((D, D, D, 4), np.float32)
            host[1:-1, 1:-1, 1:-1] = level0
        A.call("vct_dense_write_level", h, None, 0, host.ctypes.data_as(C.c_void_p), host.nbytes)
        A.call("vct_dense_mipmap", h, None)
        for m, ref in enumerate(_mips(level0, fmt), 1):
            n = (res >> m) + 2
            got = np.empty((6, n, n, n) + ((4,) if fmt == O.FMT_RGBA32F else ()), host.dtype)
            A.call("vct_dense_read_level", h, None, m, got.ctypes.data_as(C.c_void_p), got.nbytes)
            want = np.zeros_like(got)
            if fmt == O.FMT_RGBA8:
                ref = (ref << np.arange(0, 32, 8, dtype=np.uint32)).sum(-1, dtype=np.uint32)
            want[:, 1:-1, 1:-1, 1:-1] = ref
            np.testing.assert_array_equal(got, want, err_msg=f"level {m}")
    finally:
        A.call("vct_dense_destroy", h)


@pytest.mark.parametrize("brick", [4, 8])
def test_batched_mips_equal_per_scene_ones(brick):
    """Grids of 8^3 to 128^3 in one batch: the brick shapes and the tail."""
    import torch
    import vk_voxel_cone_tracing_amd as V
    from vk_voxel_cone_tracing_amd import scenes, workloads

    A, sc, items = V._abi, workloads.scratch_ctx(), []
    for i, res in enumerate((8, 16, 32, 128)):
        scene = scenes.room(i, n_boxes=8, n_spheres=1)
        ds, cam = V.DeviceScene(scene), scenes.camera(i, 24, 16)
        gmin, ext = workloads.grid_box(scene)
        items.append(dict(ds=ds, res=res, gb=V.gbuffer_struct(workloads.gbuffer(sc, ds, scene, cam, 24, 16)),
                          cam=V.camera_ubo(*cam), gmin=gmin, ext=ext, out=torch.zeros((16, 24, 4), device="cuda")))
    A.call("vct_destroy", sc)
    td = workloads.dense_trace_desc(1.7)
    b = C.c_void_p()
    A.call("vct_batch_create", C.byref(b), workloads.batch_scene_array(items), len(items), C.byref(td))
    A.call("vct_batch_set_tuning", b, C.byref(A.BatchTuning(256, brick, 0, 0)))
    for _ in range(2):  # the second run starts from the winners the first returned to empty
        A.call("vct_batch_run", b, C.c_void_p(torch.cuda.current_stream().cuda_stream), None)
    A.call("vct_batch_status", b)
    for i, it in enumerate(items):
        h = C.c_void_p()
        A.call("vct_dense_create", C.byref(h),
               C.byref(A.DenseDesc(A.f3(*it["gmin"]), it["ext"], it["res"], 0, 1, 0)))
        A.call("vct_dense_voxelize", h, None, C.byref(it["ds"].mesh))
        A.call("vct_dense_mipmap", h, None)
        for m in range(it["res"].bit_length()):
            n = ((it["res"] >> m) + 2) ** 3 * (6 if m else 1)
            one, got = np.empty(n, np.uint32), np.empty(n, np.uint32)
            A.call("vct_dense_read_level", h, None, m, one.ctypes.data_as(C.c_void_p), one.nbytes)
            A.call("vct_batch_read_level", b, None, i, m, got.ctypes.data_as(C.c_void_p), got.nbytes)
            np.testing.assert_array_equal(got, one, err_msg=f"scene {i} level {m}")
        A.call("vct_dense_destroy", h)
    A.call("vct_batch_destroy", b)
