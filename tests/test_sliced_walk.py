"""The walk of a streamed cast (bricks put off and walked in slices), which on the
device runs for every large ray array, on the CPU: the same result and the same
count of iterations as cast_ray and cast_ray_lod, under every iteration bound."""
from __future__ import annotations

import numpy as np
import pytest

import hostsim
from shocovox_amd import Octree, workloads as W

LIMITS = (0, 1, 2, 5, 9, 17, 40, 200)  # (0: the default bound)


def _rays(size: int, n: int) -> np.ndarray:
    rays = W.incoherent_rays(size, n, seed=size + n)
    rays[::4, :3] -= rays[::4, 3:] * np.float32(1.5 * size)
    rays[0, 3:] = (0.0, 0.0, 1.0)
    rays[1, 3:] = (-1.0, 0.0, 0.0)
    rays[2, 3] = np.inf
    rays[3, 4] = np.nan
    rays[5, 3:] = 0.0
    return rays


@pytest.mark.parametrize("kind,size,dim", [(2, 64, 1), (2, 64, 2), (2, 64, 8), (1, 128, 16),
                                           (3, 128, 32), (4, 64, 4)])
@pytest.mark.parametrize("sliced", [1, 3, 20])
def test_sliced_walk_equals_the_plain_one(kind, size, dim, sliced):
    tree = Octree.scene(kind, size, dim, 4)
    tree.albedo_mip_map_resampling_strategy().switch_albedo_mip_maps(True).recalculate_mips()
    a = tree.flatten().arrays()
    rays = _rays(size, 400)
    guarded = 0
    for limit in LIMITS:
        for vd in (None, 0.3 * size, 4.0 * size):
            few = rays if limit else rays[6:]  # (a NaN ray runs into any bound)
            with np.errstate(all="ignore"):
                want = hostsim.cast(a, few, max_steps=limit, viewing_distance=vd)
                got = hostsim.cast(a, few, max_steps=limit, viewing_distance=vd, sliced=sliced)
            assert want.tobytes() == got.tobytes(), (limit, vd)
            guarded += int((want["flags"] & 1).sum())
    assert guarded > 0 and int((want["hit"] == 1).sum()) > 0
