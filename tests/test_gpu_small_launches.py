"""Plain launches of few rays, whose waves take fewer than 64 of them each:
ray counts and image shapes on both sides of every split, against the oracle
(bit for bit)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from parity import assert_parity, gpu_to_numpy
from shocovox_amd import DeviceTree, Octree, workloads as W

pytestmark = pytest.mark.gpu

SPLITS = [2048 << k for k in range(2, 7)]  # rays up to which waves take 4, 8, .. 64


@pytest.fixture(scope="module")
def scene(gpu_device):
    tree = Octree.scene(2, 128, 8, 3)
    tree.albedo_mip_map_resampling_strategy().switch_albedo_mip_maps(True).recalculate_mips()
    return DeviceTree(tree), oracle.OracleTree(tree.export_model())


@pytest.mark.parametrize("n", [1, 3, 5] + [s + e for s in SPLITS for e in (0, 1)])
def test_casts(scene, gpu_device, n):
    import torch
    dtree, otree = scene
    print(f"cast of {n} rays", flush=True)
    rays = W.incoherent_rays(128, n, seed=n)
    dev = torch.from_numpy(rays).to(gpu_device)
    got, lod = dtree.cast(dev), dtree.cast_at_lod(dev, 64.0)
    torch.cuda.synchronize()
    assert_parity(otree.cast(rays), gpu_to_numpy(got), f"{n} rays")
    assert_parity(otree.cast(rays, viewing_distance=64.0), gpu_to_numpy(lod), f"{n} LOD rays")


@pytest.mark.parametrize("w,h", [(1, 1), (1, 9), (5, 3), (8192, 1), (1, 8193), (127, 129),
                                 (255, 129), (256, 256), (263, 251), (511, 257)])
def test_frames(scene, w, h):
    import torch
    dtree, otree = scene
    print(f"frame of {w}x{h}", flush=True)
    vp = W.look_at_viewport((180.0, 150.0, -30.0), (64.0, 50.0, 64.0), w, h)
    rays = oracle.viewport_rays(vp.origin, vp.direction, vp.frustum, vp.fov, w, h)
    got, lod = dtree.render(vp, w, h), dtree.render_at_lod(vp, w, h, 64.0)
    shaded = [dtree.render_rgba8(vp, w, h, c) for c in (0, 1)]
    torch.cuda.synchronize()
    exp = otree.cast(rays)
    assert_parity(exp, gpu_to_numpy(got), f"{w}x{h}")
    assert_parity(otree.cast(rays, viewing_distance=64.0), gpu_to_numpy(lod), f"{w}x{h} LOD")
    # (the shading itself is tested elsewhere: here, that every pixel is written)
    for image in shaded:
        assert ((image.cpu().numpy().view(np.uint32) >> 24) == 0xFF).all()
