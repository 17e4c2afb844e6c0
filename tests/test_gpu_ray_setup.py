"""A ray's setup on the device divides and takes roots without the handling of
extreme exponents where its operands are far from them: directions and origins
on both sides of every such limit, against the oracle (bit for bit).
Directions that are not of unit length are compared with the host build of the
same traversal, whose quotients and roots are the host's: its power-of-two form
differs from the oracle in the last bit of an impact for a few such rays."""
from __future__ import annotations

import numpy as np
import pytest

import hostsim
import oracle
from parity import assert_parity, gpu_to_numpy
from shocovox_amd import DeviceTree, Octree, workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def scene(gpu_device):
    tree = Octree.scene(2, 64, 4, 3)
    return (DeviceTree(tree), oracle.OracleTree(tree.export_model()), tree.flatten().arrays())


def _check(scene, gpu_device, rays, label, unit=True):
    import torch
    dtree, otree, layout = scene
    print(label, flush=True)
    got = dtree.cast(torch.from_numpy(np.ascontiguousarray(rays)).to(gpu_device))
    torch.cuda.synchronize()
    with np.errstate(all="ignore"):
        exp = otree.cast(rays, threads=8) if unit else hostsim.cast(layout, rays)
    assert_parity(exp, gpu_to_numpy(got), label)


@pytest.mark.parametrize("power", [-8, -4, -1, 0, 1, 12, 23, 24, 25, 40, 61])
def test_lengths_of_directions(scene, gpu_device, power):
    rays = W.incoherent_rays(64, 4000, seed=power + 100)
    rays[::2, :3] -= rays[::2, 3:] * np.float32(100.0)
    rays[:, 3:] *= np.float32(2.0 ** power)
    _check(scene, gpu_device, rays, f"directions of length 2^{power}", unit=False)


@pytest.mark.parametrize("power", [-23, -24, -25, -40, -60, -61, -130])
def test_small_components(scene, gpu_device, power):
    rays = W.incoherent_rays(64, 3000, seed=power + 200)
    for axis in range(3):
        rays[axis::6, 3 + axis] = np.float32(2.0 ** power) * np.sign(rays[axis::6, 3 + axis])
    _check(scene, gpu_device, rays, f"a direction component of 2^{power}")
    # an origin as far from one face of the tree
    rays = W.incoherent_rays(64, 3000, seed=power + 300)
    for axis in range(3):
        rays[axis::3, axis] = np.float32(2.0 ** power)
        rays[axis::12, axis] = -np.float32(2.0 ** power)
        rays[axis::9, axis] = 0.0
    _check(scene, gpu_device, rays, f"an origin 2^{power} from a face")


def test_far_origins(scene, gpu_device):
    rays = W.incoherent_rays(64, 4000, seed=7)
    away = np.float32(2.0) ** np.linspace(3, 70, len(rays), dtype=np.float32)
    with np.errstate(over="ignore"):
        rays[:, :3] -= rays[:, 3:] * away[:, None]
    _check(scene, gpu_device, rays, "origins up to 2^70 away")
