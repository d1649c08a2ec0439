"""GPU SpecularFilterPass at the edges of its tiles: images smaller than a
tile, one past it, a tall narrow one, and one large enough for the four-row
bilateral kernel (512 workgroups of 64 x 16 pixels)."""
import ctypes as C

import numpy as np
import pytest

import oracle_api as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("method", [1, 0])
@pytest.mark.parametrize("W,H", [(1, 1), (3, 2), (64, 4), (65, 17), (7, 130), (2049, 257)])
def test_specular_filter_sizes(W, H, method):
    import torch
    import vk_voxel_cone_tracing_amd as V

    rng = np.random.default_rng(W * 1000 + H)
    diffuse = rng.uniform(0, 2, (H, W, 4)).astype(np.float32)
    spec = rng.uniform(0, 1, (H, W, 4)).astype(np.float32)
    d_t, s_t = torch.from_numpy(diffuse).cuda(), torch.from_numpy(spec).cuda()
    out = torch.empty_like(d_t)
    desc = V._abi.SpecularFilterDesc(2.2, 0.1, 0, method)
    V._abi.call("vct_specular_filter", None, C.c_void_p(d_t.data_ptr()), C.c_void_p(s_t.data_ptr()), W, H,
                C.byref(desc), C.c_void_p(out.data_ptr()))
    torch.cuda.synchronize()
    ref = O.specular_filter(diffuse, spec, 2.2, 0.1, 0, method)
    # The oracle's taps sit at FP32 texture coordinates: one is rounded by at
    # most 2^-23 (coordinate and offset sum), i.e. 2^-23 size texels, and its
    # product with the size by as much again; a bilinear tap moves by at most
    # the texel range per texel and axis (2 for the diffuse image, 1 for the
    # specular one). 2e-6 relative covers the FP32 sums.
    atol = 2 * 2.0 ** -23 * (W + H) * 3 + 2e-6
    np.testing.assert_allclose(out.cpu().numpy(), ref, rtol=2e-6, atol=atol)
