"""The clipmap trace's splits by image size against the oracle: sixteen waves
per 8x8 tile and sixteen lanes per specular cone for the smallest images, four
waves and four lanes for larger ones, with edge tiles cut by the image border,
in modes with and without the specular pass and the direct term."""
import pytest

import test_gpu_clipmap as clipmap

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,mode,cones32,W,H", [
    (1, 6, 0, 33, 17),     # 16 lanes, no diffuse cones
    (0, 8, 1, 121, 71),    # 16 lanes, 16 waves, 32 cones
    (1, 8, 0, 203, 101),   # 20503 pixels: 4 lanes; 364 tiles: 4 waves
    (0, 5, 1, 203, 101),   # direct term without a specular pass
])
def test_split_trace_matches_oracle(fmt, mode, cones32, W, H):
    clipmap.test_trace_matches_oracle(fmt, mode, cones32, W, H, 32, 3)
