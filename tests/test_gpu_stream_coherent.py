"""Streamed casts of rays that belong together: camera rays in rows of pixels and
in 8x8 tiles, alone and in turn with random ones, against the oracle (bit for
bit) and, as to time, against a render of the same view."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from parity import assert_parity, gpu_to_numpy
from shocovox_amd import Batch, DeviceTree, Octree, alloc_hits, workloads as W

pytestmark = pytest.mark.gpu

FIELDS = ("hit", "albedo", "voxel", "distance")


def _tiles(w: int, h: int) -> np.ndarray:
    """Pixel numbers of a w x h image (multiples of 8) in order of 8x8 tiles."""
    return np.arange(w * h).reshape(h // 8, 8, w // 8, 8).transpose(0, 2, 1, 3).reshape(-1)


@pytest.mark.parametrize("order", ["rows", "tiles", "in turn"])
@pytest.mark.parametrize("cut", [0, 1, 63, 64 * 1000 + 31])
def test_camera_rays(gpu_device, order, cut):
    import torch
    size, w, h = 128, 1024, 896
    tree = Octree.scene(2, size, 8, 5)
    tree.albedo_mip_map_resampling_strategy().switch_albedo_mip_maps(True).recalculate_mips()
    otree, dtree = oracle.OracleTree(tree.export_model()), DeviceTree(tree)
    vp = W.look_at_viewport((180.0, 150.0, -30.0), (64.0, 50.0, 64.0), w, h)
    rays = oracle.viewport_rays(vp.origin, vp.direction, vp.frustum, vp.fov, w, h)
    if order != "rows":
        rays = rays[_tiles(w, h)]
    if order == "in turn":  # groups of 64: near each other, random, half and half
        other = W.incoherent_rays(size, len(rays), seed=4).reshape(-1, 64, 6)
        groups = rays.reshape(-1, 64, 6)
        groups[1::3] = other[1::3]
        groups[2::3, ::2] = other[2::3, ::2]
        groups[3::30, 0, 3:] = np.inf
        rays = groups.reshape(-1, 6)
    rays = np.ascontiguousarray(rays[: len(rays) - cut])
    dev = torch.from_numpy(rays).to(gpu_device)
    print(f"{len(rays)} camera rays, {order}", flush=True)
    got, lod = dtree.cast(dev), dtree.cast_at_lod(dev, 90.0)
    torch.cuda.synchronize()
    with np.errstate(all="ignore"):
        assert_parity(otree.cast(rays, threads=8), gpu_to_numpy(got), order)
        assert_parity(otree.cast(rays, viewing_distance=90.0, threads=8), gpu_to_numpy(lod),
                      f"{order} at LOD")


def test_cast_of_a_frame_takes_about_a_frame(gpu_device):
    """8.3M camera rays in tiles, as an array, against a render of them: with runs
    of neighbouring rays dealt to each wave the launch lasted 4.8 times the
    one-ray-per-lane kernel's time on caves 512^3 and 10.5 times on heights 256^3,
    dealt in groups a grid apart 1.6 and 1.4 times. 2.5 lies well between."""
    import torch
    w, h = 3840, 2160
    order = torch.from_numpy(_tiles(w, h)).to(gpu_device)
    for kind, size, dim in ((2, 512, 16), (4, 256, 8)):
        dtree = DeviceTree(Octree.scene(kind, size, dim, 5))
        vp = W.look_at_viewport((1.4 * size, 0.8 * size, -0.2 * size), (size / 2, 0.4 * size,
                                                                        size / 2), w, h)
        rays = oracle.viewport_rays(vp.origin, vp.direction, vp.frustum, vp.fov, w, h)
        rays = torch.from_numpy(rays).to(gpu_device)[order].contiguous()
        image, hits = (alloc_hits(w * h, gpu_device, FIELDS) for _ in range(2))

        def micros(call):
            best = float("inf")
            for _ in range(6):
                a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
                a.record()
                call()
                b.record()
                torch.cuda.synchronize()
                best = min(best, a.elapsed_time(b) * 1e3)
            return best

        frame = micros(lambda: dtree.render_into(vp, w, h, image))
        cast = micros(lambda: dtree.cast_into(rays, w * h, hits))
        print(f"{size}^3/{dim}: frame {frame:.0f} us, cast {cast:.0f} us", flush=True)
        for k in FIELDS:
            v = image[k].reshape(w * h, -1)[order]
            assert torch.equal(v, hits[k].reshape(w * h, -1)), k
        assert cast < 2.5 * frame


def test_large_jobs_of_one_run_overlap(gpu_device):
    """Four 720p arrays in one run: as streamed casts one after another they took
    what four calls take, as tiles of one launch less than half of it; 0.75 lies
    between. With a job of more than 2^20 rays, which is streamed, results are
    those of plain calls too."""
    import torch
    size, w, h = 512, 1280, 720
    dtree = DeviceTree(Octree.scene(2, size, 16, 5))
    order = torch.from_numpy(_tiles(w, h)).to(gpu_device)
    arrays = []
    for i in range(4):
        vp = W.look_at_viewport((1.4 * size, 0.8 * size, (i - 1.2) * 0.3 * size),
                                (size / 2, 0.4 * size, size / 2), w, h)
        rays = oracle.viewport_rays(vp.origin, vp.direction, vp.frustum, vp.fov, w, h)
        arrays.append(torch.from_numpy(rays).to(gpu_device)[order].contiguous())
    arrays.append(torch.from_numpy(W.incoherent_rays(size, (1 << 20) + 77, 3)).to(gpu_device))
    want = [dtree.cast(r, FIELDS) for r in arrays]
    outs = [alloc_hits(len(r), gpu_device, FIELDS) for r in arrays]
    for n in (4, 5):
        for o in outs:
            for v in o.values():
                v.fill_(-3)
        batch = Batch(n)
        jobs = [Batch.cast_job(dtree, r, o) for r, o in zip(arrays[:n], outs)]
        times = [], []
        for _ in range(6):
            for calls, t in ((lambda: batch.run(jobs), times[0]),
                             (lambda: [dtree.cast_into(r, len(r), o)
                                       for r, o in zip(arrays[:n], want)], times[1])):
                a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
                a.record()
                calls()
                b.record()
                torch.cuda.synchronize()
                t.append(a.elapsed_time(b) * 1e3)
        run, each = min(times[0]), min(times[1])
        print(f"{n} jobs: one run {run:.0f} us, {n} casts {each:.0f} us", flush=True)
        for i in range(n):
            for k in FIELDS:
                assert torch.equal(outs[i][k], want[i][k]), (i, k)
        assert n > 4 or run < 0.75 * each
