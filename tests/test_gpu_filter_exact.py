"""The specular blur against the same taps in 64 bits, at sizes where a texel's
centre is no FP32 texture coordinate (1920 wide, 8200 high): the filter's error
is that of its nine FP32 products and sums, not of the taps' coordinates."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _blur64(spec):
    """filter.glsl:9-24: the centre and 32 directions x 8 rings of bilinear taps
    up to 0.01 texel away, clamped to the edge, over 8 * 32 - 15."""
    f = np.float32
    H, W, _ = spec.shape
    p = np.pad(spec.astype(np.float64), ((1, 1), (1, 1), (0, 0)), mode="edge")
    taps = [(0.0, 0.0)]
    a, two_pi = f(0), f(6.28318530718)
    while a < two_pi:  # the shader's loops run on float accumulators
        for ring in range(1, 9):
            taps.append((np.cos(float(a)) * 0.01 * ring / 8, np.sin(float(a)) * 0.01 * ring / 8))
        a = f(a + two_pi / f(32))
    w = np.zeros((3, 3))
    for dx, dy in taps:
        w += np.outer([max(-dy, 0), 1 - abs(dy), max(dy, 0)], [max(-dx, 0), 1 - abs(dx), max(dx, 0)])
    return sum(w[j, i] / (8 * 32 - 15) * p[j:j + H, i:i + W] for j in range(3) for i in range(3))


@pytest.mark.parametrize("W,H", [(1920, 40), (5, 8200)])
def test_blur_is_its_taps_in_64_bits(W, H):
    import torch
    import vk_voxel_cone_tracing_amd as V

    spec = np.random.default_rng(W).uniform(0, 1, (H, W, 4)).astype(np.float32)
    s_t = torch.from_numpy(spec).cuda()
    d_t, out = torch.zeros_like(s_t), torch.empty_like(s_t)
    desc = V._abi.SpecularFilterDesc(2.2, 0.1, 0, 1)
    V._abi.call("vct_specular_filter", None, C.c_void_p(d_t.data_ptr()), C.c_void_p(s_t.data_ptr()), W, H,
                C.byref(desc), C.c_void_p(out.data_ptr()))
    torch.cuda.synchronize()
    got, ref = out.cpu().numpy()[..., :3], _blur64(spec)[..., :3]
    # weights and products rounded once each and at most eight sums, all terms
    # positive: 10 roundings of 2^-24 relative
    np.testing.assert_allclose(got, ref, rtol=10 * 2.0 ** -24, atol=0)
