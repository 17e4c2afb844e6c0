"""The per-tile batched kernel (variant "auto"): job counts on both sides of
its 64-job search blocks, empty jobs, images one tile wide, runs small enough
that a wave takes part of a tile; against plain launches of the same jobs,
which other tests compare with the oracle (bit for bit)."""
from __future__ import annotations

import numpy as np
import pytest

from shocovox_amd import (Batch, DeviceTree, Octree, alloc_hits, batch_variants,
                          current_batch_variant, workloads as W)

pytestmark = pytest.mark.gpu

SHAPES = [(8, 8), (1, 70), (33, 17), (0, 5), (64, 1), (7, 9)]


@pytest.mark.parametrize("njobs,scale,vd", [(1, 1, 0.0), (1, 24, 0.0), (2, 9, 32.0), (63, 1, 0.0),
                                            (64, 1, 16.0), (65, 3, 0.0), (200, 5, 0.0)])
def test_jobs_equal_plain_launches(gpu_device, njobs, scale, vd):
    import torch
    assert batch_variants()[current_batch_variant()] == "auto"
    print(f"{njobs} jobs, images x{scale}, viewing distance {vd}", flush=True)
    dtrees = []
    for size, dim, seed in ((64, 4, 1), (128, 8, 2)):
        t = Octree.scene(2, size, dim, seed)
        t.albedo_mip_map_resampling_strategy().switch_albedo_mip_maps(True).recalculate_mips()
        dtrees.append((size, DeviceTree(t)))
    batch = Batch(njobs)
    jobs, pairs = [], []
    for i in range(njobs):
        size, d = dtrees[i % 2]
        lod = vd if i % 3 == 0 else 0.0
        if i % 5 == 4:
            n = 37 * scale * (i % 7)
            rays = torch.from_numpy(W.incoherent_rays(size, n, seed=i)).to(gpu_device)
            out = alloc_hits(n, gpu_device)
            jobs.append(Batch.cast_job(d, rays, out, lod))
            want = d.cast_at_lod(rays, lod) if lod else d.cast(rays)
        else:
            w, h = (v * scale for v in SHAPES[i % len(SHAPES)])
            if njobs == 1:
                w, h = 33 * scale, 17 * scale
            vp = W.look_at_viewport((1.4 * size, size, -0.3 * size + i), (size / 2,) * 3,
                                    max(w, 1), max(h, 1))
            out = alloc_hits(w * h, gpu_device)
            jobs.append(Batch.render_job(d, vp, w, h, out, lod))
            want = d.render_at_lod(vp, w, h, lod) if lod else d.render(vp, w, h)
        pairs.append((out, want))
    for rnd in range(2):  # (the second run overwrites the first's table)
        for out, _ in pairs:
            for v in out.values():
                v.fill_(-3)
        batch.run(jobs)
        torch.cuda.synchronize()
        for i, (out, want) in enumerate(pairs):
            for k in out:
                a, b = (x[k].cpu().numpy() for x in (out, want))
                assert a.tobytes() == b.tobytes(), f"run {rnd}, job {i}, {k}"
    assert sum(int((np.asarray(o["hit"].cpu()) == 1).sum()) for o, _ in pairs) > 0
