"""Injection records piled up on one texel: 600 overlapping quads (300 facing
each way), quad k covering the first k / 300 of the floor's width, so the
runs of records per texel take every length from 1 to 300, past a wave, two
waves and the 256 at which the RGBA8 count wraps; bit for bit against the
oracle. One quad has zero normals (its radiance is not a number)."""
import ctypes as C

import numpy as np
import pytest

import oracle_api as O
import test_gpu_clipmap as clipmap

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,nan_normals", [(0, False), (1, False), (0, True)])
def test_long_runs_bit_exact(fmt, nan_normals):
    import torch
    import vk_voxel_cone_tracing_amd as V
    from vk_voxel_cone_tracing_amd import scenes

    S, K = clipmap.SCALE, 300
    b = scenes._Builder()
    rng = np.random.default_rng(4)
    for k in range(K):
        w = S * (k + 1) / K
        for up in (1.0, -1.0):
            P = np.array([(0, 2.03, 0), (w, 2.03, 0), (w, 2.03, S), (0, 2.03, S)], np.float32)
            n = (0.3, up, 0.2) if not (nan_normals and k == 7) else (0.0, 0.0, 0.0)
            ref = b.mesh(P, np.tile(np.array(n, np.float32), (4, 1)), np.array([0, 1, 2, 0, 2, 3], np.uint32))
            em = tuple(rng.uniform(0.1, 1, 3)) if k % 41 == 40 else (0.0, 0.0, 0.0)
            b.draw(ref, np.eye(4), scenes._material(rng.uniform(0.2, 0.8, 3), em), scenes._surface(rng))
    scene = b.build(1.0)
    res, levels = clipmap.RES, clipmap.LEVELS
    ctx = V.Context(resolution=res, levels=levels, radiance_format=fmt, downsample_region_size=2,
                    extent_l0=clipmap.EXTENT_L0)
    ctx.update_clip_regions(np.full(3, 0.5 * S))
    ds = V.DeviceScene(scene)
    pos, nrm, mat = scene.world_triangles()
    light = scenes.light(0, scale=S)
    depth = np.random.default_rng(5).uniform(0.2, 1, (64, 64)).astype(np.float32)
    ld, ls = V.light_structs(light)
    sm = V.shadow_struct(torch.from_numpy(depth).cuda())
    ctx.clear_volume(V.VOLUME_RADIANCE)
    ref = O.new_volume(res, levels, fmt)
    osm, olight = O.Shadow(depth.ctypes.data, 64, 64), O.light_struct(light)
    descs = [ctx.voxelization_desc(level) for level in range(levels)]
    ctx.inject_radiance_levels(ds, sm, ld, ls, descs)
    for level, desc in enumerate(descs):
        O.lib().orc_inject_radiance(C.byref(O.vol_struct(ref, res, levels)), C.byref(O.tris_struct(pos, nrm, mat)),
                                    O.materials_struct(scene), C.byref(osm), C.byref(olight),
                                    C.byref(clipmap._desc_to_oracle(desc, ctx.regions[level])), 1, 0x3F)
    assert int((ref != 0).sum()) > 1000
    np.testing.assert_array_equal(ctx.read_volume(V.VOLUME_RADIANCE), ref)
