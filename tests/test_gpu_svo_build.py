"""The octree build at the widths of its sorted paths (30 bits at level 10, 33
bits at level 11, 3 bits at level 1) and at fragment counts from a few to past
several workgroups of 1024: small triangles scattered over the box, some of
them stacked so that leaves average many fragments. Pool and fragments are bit
for bit the oracle's."""
import numpy as np
import pytest

import test_gpu_svo as svo

pytestmark = pytest.mark.gpu


def _scattered(n, size):
    from vk_voxel_cone_tracing_amd import scenes

    b = scenes._Builder()
    rng = np.random.default_rng(n)
    corners = [np.zeros(3), np.ones(3)]
    for k in range(n):
        at = corners[k] if k < 2 else rng.uniform(0.1, 0.9, 3)
        tri = np.array([[0, 0, 0], [1, 0.1, 0], [0.1, 1, 0.2]]) * size * (1 if k % 2 == 0 else -1)
        for _ in range(1 if k % 5 else 7):
            ref = b.mesh((at + tri).astype(np.float32), np.tile(np.array([0.3, 1, 0.2], np.float32), (3, 1)),
                         np.arange(3, dtype=np.uint32))
            b.draw(ref, np.eye(4), scenes._material(rng.uniform(0.2, 0.8, 3)), scenes._surface(rng))
    return b.build(1.0)


@pytest.mark.parametrize("level,n,size,quirks", [(1, 30, 0.8, 0x00), (4, 30, 0.1, 0x3F), (10, 2, 0.01, 0x00),
                                                 (10, 40, 0.02, 0x3F), (11, 2, 0.01, 0x3F), (11, 60, 0.02, 0x00)])
def test_pool_bit_exact(level, n, size, quirks, monkeypatch):
    monkeypatch.setattr(svo, "_scene", lambda: _scattered(n, size))
    r = svo._run(quirks, level=level)
    print(f"level {level}: {len(r['frags'])} fragments, {len(r['nodes'])} nodes")
    assert len(r["frags"]) > 0
    np.testing.assert_array_equal(r["frags"], r["ofrags"])
    np.testing.assert_array_equal(r["nodes"], r["onodes"])
