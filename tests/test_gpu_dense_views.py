"""vct_dense_trace_views: several views in one call give the images and tapes
of one call per view, bit for bit: more views than a launch takes, edge tiles,
sixteen and four waves per tile (the one call sees more tiles than each view
alone, so the two sides take different splits)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H,views,cones32", [(9, 7, 17, 0), (200, 60, 3, 1), (130, 97, 2, 0)])
def test_views_equal_single_calls(W, H, views, cones32):
    import torch
    import vk_voxel_cone_tracing_amd as V
    from vk_voxel_cone_tracing_amd import scenes, workloads

    A, res = V._abi, 32
    scene = scenes.room(1, n_boxes=12, n_spheres=2)
    ds, sc = V.DeviceScene(scene), workloads.scratch_ctx()
    cams3 = [scenes.camera(50 + v, W, H) for v in range(views)]
    gs = [workloads.gbuffer(sc, ds, scene, c, W, H) for c in cams3]
    A.call("vct_destroy", sc)
    gen = torch.Generator(device="cuda").manual_seed(3)
    albedo = torch.rand((res, res, res, 3), generator=gen, device="cuda")
    opacity = torch.rand((res, res, res), generator=gen, device="cuda") * 0.4
    h = C.c_void_p()
    A.call("vct_dense_create", C.byref(h), C.byref(A.DenseDesc(A.f3(0, 0, 0), 1.0, res, 2, 1, 0)))
    ptr = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
    A.call("vct_dense_set_level0", h, None, ptr(albedo), ptr(opacity))
    A.call("vct_dense_mipmap", h, None)
    td = workloads.dense_trace_desc(1.7)
    td.enable_32_cones = cones32
    gbs, cams = (A.GBuffer * views)(*[V.gbuffer_struct(g) for g in gs]), (A.CameraUBO * views)(*[V.camera_ubo(*c) for c in cams3])
    n = C.c_size_t()
    A.call("vct_dense_tape_bytes", h, C.byref(gbs[0]), C.byref(cams[0]), C.byref(td), C.byref(n))
    buf = lambda *s, **k: [torch.zeros(s, device="cuda", **k) for _ in range(views)]  # noqa: E731
    one, one_tape, plain = buf(H, W, 4), buf(n.value, dtype=torch.uint8), buf(H, W, 4)
    got, got_tape = buf(H, W, 4), buf(n.value, dtype=torch.uint8)
    for v in range(views):
        A.call("vct_dense_trace_tape", h, None, C.byref(gbs[v]), C.byref(cams[v]), C.byref(td), ptr(one[v]), None,
               ptr(one_tape[v]), n.value)
    ptrs = lambda ts: (C.c_void_p * views)(*[t.data_ptr() for t in ts])  # noqa: E731
    A.call("vct_dense_trace_views", h, None, views, gbs, cams, C.byref(td), ptrs(got), ptrs(got_tape), n.value)
    A.call("vct_dense_trace_views", h, None, views, gbs, cams, C.byref(td), ptrs(plain), None, 0)
    torch.cuda.synchronize()
    for v in range(views):
        np.testing.assert_array_equal(got[v].cpu().numpy(), one[v].cpu().numpy())
        np.testing.assert_array_equal(plain[v].cpu().numpy(), one[v].cpu().numpy())
        assert torch.equal(got_tape[v], one_tape[v])
    with pytest.raises(V.VctError):
        A.call("vct_dense_trace_views", h, None, views, gbs, cams, C.byref(td), ptrs(got), ptrs(got_tape), n.value - 1)
    A.call("vct_dense_destroy", h)
