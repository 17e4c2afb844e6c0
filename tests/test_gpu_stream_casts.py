"""Streamed casts (ray arrays larger than the lanes that run at once): counts
on both sides of the line and with every kind of remainder, plain and at LOD,
alone and as a batched job, against the oracle (bit for bit)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from parity import assert_parity, gpu_to_numpy
from shocovox_amd import Batch, DeviceTree, Octree, alloc_hits, workloads as W

pytestmark = pytest.mark.gpu

LINE = 6 * 1024 * 64  # rays beyond which svo_cast streams (twice as many for LOD rays)


def _rays(size: int, n: int, seed: int) -> np.ndarray:
    """Incoherent rays, some axis-aligned or infinite, some from outside the
    tree. (A NaN direction runs into the iteration bound on every side.)"""
    rays = W.incoherent_rays(size, n, seed)
    rays[::1001, 3:] = (0.0, 0.0, 1.0)
    rays[11::1777, 3] = np.inf
    rays[::5, :3] -= rays[::5, 3:] * np.float32(1.5 * size)
    return np.ascontiguousarray(rays)


@pytest.mark.parametrize("kind,size,dim,n", [(2, 128, 8, LINE), (2, 128, 8, LINE + 1),
                                             (2, 64, 4, LINE + 6143), (3, 256, 32, 460_003),
                                             (4, 256, 16, 2 * LINE), (2, 64, 2, 2 * LINE + 1),
                                             (2, 128, 8, 2 * LINE + 1)])
def test_casts(gpu_device, kind, size, dim, n):
    import torch
    tree = Octree.scene(kind, size, dim, 5)
    mips = size <= 128
    if mips:
        tree.albedo_mip_map_resampling_strategy().switch_albedo_mip_maps(True).recalculate_mips()
    otree, dtree = oracle.OracleTree(tree.export_model()), DeviceTree(tree)
    rays = _rays(size, n, seed=n)
    dev = torch.from_numpy(rays).to(gpu_device)
    print(f"scene {kind} {size}^3/{dim}, {n} rays", flush=True)
    got = dtree.cast(dev)
    torch.cuda.synchronize()
    with np.errstate(all="ignore"):
        exp = otree.cast(rays, threads=8)
    assert_parity(exp, gpu_to_numpy(got), f"{n} rays")
    if mips:
        print("at LOD", flush=True)
        lod = dtree.cast_at_lod(dev, 0.7 * size)
        torch.cuda.synchronize()
        assert_parity(otree.cast(rays, viewing_distance=0.7 * size, threads=8),
                      gpu_to_numpy(lod), f"{n} LOD rays")


def test_batched_jobs_among_others(gpu_device):
    import torch
    tree = Octree.scene(2, 128, 8, 6)
    tree.albedo_mip_map_resampling_strategy().switch_albedo_mip_maps(True).recalculate_mips()
    dtree = DeviceTree(tree)
    big = torch.from_numpy(_rays(128, 2 * LINE + 77, 1)).to(gpu_device)
    small = big[:999].contiguous()
    vp = W.look_at_viewport((180.0, 150.0, -30.0), (64.0, 50.0, 64.0), 90, 70)
    outs = [alloc_hits(k, gpu_device) for k in (len(big), 6300, len(big), 999)]
    batch = Batch(4)
    print("two streamed jobs, a render and a small cast in one run", flush=True)
    batch.run([Batch.cast_job(dtree, big, outs[0]), Batch.render_job(dtree, vp, 90, 70, outs[1]),
               Batch.cast_job(dtree, big, outs[2], 90.0), Batch.cast_job(dtree, small, outs[3])])
    assert batch.tiles == 2 * (-(-len(big) // 64)) + 12 * 9 + 16
    want = [dtree.cast(big), dtree.render(vp, 90, 70), dtree.cast_at_lod(big, 90.0),
            dtree.cast(small)]
    torch.cuda.synchronize()
    for i, (a, b) in enumerate(zip(outs, want)):
        for k in a:
            assert a[k].cpu().numpy().tobytes() == b[k].cpu().numpy().tobytes(), (i, k)
