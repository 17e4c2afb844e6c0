"""Which kernel a large ray array is cast by, and when its rays are sorted first:
on the CPU, with a stand-in for the HIP runtime that logs the launches."""
from __future__ import annotations

import pytest

import fakehip

CODE = """
import sys
sys.modules["torch"] = None  # (its libraries would register their kernels with the stand-in)
import ctypes as C
from shocovox_amd import DeviceTree, Octree, _native as N
L = N.lib()
F = C.CDLL({lib!r})
F.fake_log.restype = C.c_char_p
tree = DeviceTree(Octree.scene(2, 64, 4, 3))
threshold, n, want = {threshold!r}, {n!r}, {want!r}
if threshold is not None:
    assert L.svo_cast_set_order_threshold(threshold) == 0
for cast in (lambda: L.svo_cast(tree._h, 0x1000, n, C.byref(N.Hits()), 0x2000),
             lambda: L.svo_cast_at_lod(tree._h, 0x1000, n, 50.0, C.byref(N.Hits()), 0x2000)):
    F.fake_clear_log()
    assert cast() == 0
    log = [l.split() for l in F.fake_log().decode().splitlines()]
    # (the stand-in has no memory for the sort: sorted rays keep their order)
    sorts = any(l[0] == "nopool" for l in log)
    streams = any(l[0] == "launch" and "cast_stream_kernel" in l[1] for l in log)
    plain = any(l[0] == "launch" and ("11cast_kernel" in l[1] or "cast_lod_kernel" in l[1])
                for l in log)
    assert [sorts, streams, plain] == dict(sort=[True, False, True],
                                           stream=[False, True, False])[want], log
"""
M = 1 << 20


@pytest.mark.parametrize("threshold,n,want", [
    (None, M, "stream"), (None, 3 * M, "stream"), (0, M, "stream"),
    # every count is a threshold, the default's own included
    (M, M, "sort"), (M, M - 1, "stream"), (M - 1, M, "sort"), (M + 1, M, "stream"),
    (M + 1, M + 1, "sort"), (1000, 1000, "sort")])
def test_sorting_follows_the_chosen_threshold(threshold, n, want):
    fakehip.run(CODE.format(lib=str(fakehip.LIB), threshold=threshold, n=n, want=want))


BATCH = """
import sys
sys.modules["torch"] = None
import ctypes as C
from shocovox_amd import DeviceTree, Octree, _native as N
L = N.lib()
F = C.CDLL({lib!r})
F.fake_log.restype = C.c_char_p
tree = DeviceTree(Octree.scene(2, 64, 4, 3))
threshold, casts, want = {threshold!r}, {casts!r}, {want!r}
if threshold is not None:
    assert L.svo_cast_set_order_threshold(threshold) == 0
js = (N.Job * len(casts))(*[N.Job(tree._h, 1, n, 1, N.Viewport(), 0x1000, N.Hits(), vd)
                            for n, vd in casts])
b = C.c_void_p()
assert L.svo_batch_create(len(js), C.byref(b)) == 0
runs = [lambda: L.svo_batch_run(b, js, len(js), 0x2000),
        lambda: L.svo_batch_run_static(js, len(js), 0x2000)]
for i, run in enumerate(runs):
    F.fake_clear_log()
    assert run() == 0
    log = [l.split() for l in F.fake_log().decode().splitlines()]
    sorts = sum(l[0] == "nopool" for l in log) if i == 0 else want[2]  # (the static run never does)
    got = [sum(l[0] == "launch" and "cast_stream_kernel" in l[1] for l in log),
           sum(int(l[2]) for l in log if l[0] == "launch" and "batch_tile_kernel" in l[1]), sorts]
    assert got == list(want), (got, log)
L.svo_batch_destroy(b)
"""


@pytest.mark.parametrize("threshold,casts,want", [
    # alone, a job runs as svo_cast does
    (None, [(400_000, 0.0)], (1, 0, 0)), (None, [(393_216, 0.0)], (0, 6144, 0)),
    (None, [(800_000, 50.0)], (1, 0, 0)),
    # among others only from 2^20 rays: the tiles of smaller ones overlap
    (None, [(921_600, 0.0)] * 4, (0, 4 * 14400, 0)), (None, [(921_600, 50.0)] * 2, (0, 28800, 0)),
    (None, [(M - 1, 0.0), (M, 0.0), (M + 5, 50.0), (640, 0.0)], (2, 16384 + 10, 0)),
    # nor does a smaller one sort unless the caller said so
    (M, [(M - 1, 0.0), (M, 0.0)], (0, 2 * 16384, 1)), (0, [(M - 1, 0.0), (M, 0.0)], (1, 16384, 0))])
def test_large_jobs_of_a_batch(threshold, casts, want):
    fakehip.run(BATCH.format(lib=str(fakehip.LIB), threshold=threshold, casts=casts, want=want))
