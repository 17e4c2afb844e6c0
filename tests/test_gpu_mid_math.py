"""The device's reciprocal, quotient and root for operands far from extreme
exponents (svo_math.hpp) against IEEE 754 division and square root: the first
and the last rest on the hardware's estimates, which are compared for every
significand."""
from __future__ import annotations

import numpy as np
import pytest

import devmath

pytestmark = pytest.mark.gpu

F = np.float32
ALL = (np.arange(1 << 23, dtype=np.uint32) | np.uint32(127 << 23)).view(F)  # [1, 2)


def _same(got, want, label):
    a, b = got.cpu().numpy().view(np.uint32), np.asarray(want, F).view(np.uint32)
    bad = np.nonzero(a != b)[0]
    assert len(bad) == 0, f"{label}: {len(bad)} differ, first at {bad[0]}"


@pytest.mark.parametrize("power", [-24, -7, 0, 1, 23])
def test_every_reciprocal(gpu_device, power):
    import torch
    b = ALL * F(2.0 ** power)
    for sign in (F(1), F(-1)):
        print(f"1 / b, b from {sign * F(2.0 ** power)}", flush=True)
        _same(devmath.run("rcp", torch.from_numpy(b * sign).to(gpu_device)), F(1) / (b * sign),
              f"2^{power}")


@pytest.mark.parametrize("power", [-60, -59, -1, 0, 1, 60, 98, 99])
def test_every_root(gpu_device, power):
    import torch
    x = ALL * F(2.0 ** power)
    print(f"roots from 2^{power}", flush=True)
    _same(devmath.run("sqrt", torch.from_numpy(x).to(gpu_device)), np.sqrt(x), f"2^{power}")


@pytest.mark.parametrize("pa,pb", [(0, 0), (-60, 23), (-60, -24), (59, -24), (59, 23), (-5, 7),
                                   (20, -20)])
def test_quotients(gpu_device, pa, pb):
    """8.4 million pairs a range: random ones, and divisors next to powers of two
    and to the all-ones significand with every kind of numerator."""
    import torch
    rng = np.random.default_rng(100 * pa + pb + 9000)
    n = 1 << 23
    ma, mb = (rng.integers(0, 1 << 23, n, dtype=np.uint32) for _ in range(2))
    edge = np.array([0, 1, 2, 0x7FFFFF, 0x7FFFFE, 0x400000, 0x3FFFFF, 0x2AAAAA, 0x555555],
                    np.uint32)
    mb[: n // 4] = edge[rng.integers(0, len(edge), n // 4)]
    ma[: n // 16] = edge[rng.integers(0, len(edge), n // 16)]
    ma[n // 2: 5 * n // 8] = mb[n // 2: 5 * n // 8]  # quotients of a power of two
    a = (ma | np.uint32(127 << 23)).view(F) * F(2.0 ** pa)
    b = (mb | np.uint32(127 << 23)).view(F) * F(2.0 ** pb)
    a[::3] *= F(-1)
    b[::5] *= F(-1)
    a[::1000], b[::1000] = F(0), np.abs(b[::1000])
    print(f"2^{pa} / 2^{pb}", flush=True)
    _same(devmath.run("quot", torch.from_numpy(b).to(gpu_device),
                      torch.from_numpy(a).to(gpu_device)), a / b, f"2^{pa} / 2^{pb}")
