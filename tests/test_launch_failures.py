"""What batched runs answer when a launch fails, and what they keep of the work
queued before it: on the CPU, with a stand-in for the HIP runtime that logs
every call and fails the launches it is told to."""
from __future__ import annotations

import pytest

import fakehip

PRELUDE = """
import sys
sys.modules["torch"] = None  # (its libraries would register their kernels with the stand-in)
import ctypes as C
import numpy as np
from shocovox_amd import DeviceTree, Octree, _native as N, workloads as W
L = N.lib()
F = C.CDLL({lib!r})
F.fake_log.restype = C.c_char_p
F.fake_news.restype = C.c_ulong
tree = DeviceTree(Octree.scene(2, 64, 4, 3))
vp = W.look_at_viewport((90.0, 80.0, -20.0), (32.0, 30.0, 32.0), 40, 24)
rays = np.zeros(6, np.float32)  # (never read here)
BIG = (1 << 20) + 77  # rays of a job that runs by its own launch
def render():
    return N.Job(tree._h, 0, 40, 24, vp.to_c(), None, N.Hits(), 0.0)
def cast(n):
    return N.Job(tree._h, 1, n, 1, N.Viewport(), rays.ctypes.data, N.Hits(), 0.0)
def jobs(*js):
    return (N.Job * len(js))(*js)
def log():
    return [l.split() for l in F.fake_log().decode().splitlines()]
def error():
    return L.svo_last_error().decode()
S = [C.c_void_p(0x1000), C.c_void_p(0x2000)]  # (streams the stand-in only logs)
""".format(lib=str(fakehip.LIB))


@pytest.mark.parametrize("kernel", ["upload_table_kernel", "batch_tile_kernel"])
def test_static_run_reports_a_failed_launch(kernel):
    fakehip.run(PRELUDE + f"""
js = jobs(render())
assert L.svo_batch_run_static(js, 1, S[0]) == 0
F.fake_clear_log()
F.fake_fail_launch({kernel!r}.encode())
assert L.svo_batch_run_static(js, 1, S[0]) == 7, log()
assert "launch" in error(), error()
# nothing runs on a table that did not arrive
assert not any(l[0] == "launch" and "batch_tile" in l[1] for l in log()), log()
F.fake_fail_launch(b"")
assert L.svo_batch_run_static(js, 1, S[0]) == 0
""")


def test_static_run_allocates_nothing():
    """svo_batch_run_static makes no allocation on the host either, so it
    cannot run out of memory between two of its launches."""
    fakehip.run(PRELUDE + """
js = jobs(cast(BIG), render(), cast(BIG), cast(100))
for _ in range(2):
    before = F.fake_news()
    assert L.svo_batch_run_static(js, 4, S[0]) == 0
    after = F.fake_news()
assert after == before, (before, after)
""")


@pytest.mark.parametrize("small", [True, False], ids=["table-by-kernel", "table-by-copy"])
@pytest.mark.parametrize("kernel,queued", [("cast_stream_kernel", "batch_tile"),
                                           ("batch_tile_kernel", "table")])
def test_failed_run_keeps_the_work_it_queued(small, kernel, queued):
    """A run whose later launch fails has its table (and tiles) queued: the
    next run, on another stream, waits for them before it writes the device
    table, fills the other staging, and the one after that waits for this one."""
    fakehip.run(PRELUDE + f"""
small, kernel, queued = {small!r}, {kernel!r}, {queued!r}
b = C.c_void_p()
assert L.svo_batch_create(64, C.byref(b)) == 0
js = jobs(cast(BIG), *[render() for _ in range(1 if small else 60)])
def run(s):
    F.fake_clear_log()
    return L.svo_batch_run(b, js, len(js), s)
F.fake_fail_launch(kernel.encode())
assert run(S[0]) == 7, log()
F.fake_fail_launch(b"")
first = log()
table = [i for i, l in enumerate(first)
         if l[0] == "copy" or (l[0] == "launch" and "upload_table" in l[1])]
assert table and (first[table[0]][0] == "launch") == small, first
if queued == "batch_tile":
    assert any(l[0] == "launch" and queued in l[1] for l in first), first
records = [i for i, l in enumerate(first) if l[0] == "record" and l[2] == "0x1000"]
assert records and records[-1] > max(i for i, l in enumerate(first) if l[0] != "record"), first
event = first[records[-1]][1]
assert run(S[1]) == 0
second = log()
waits = [i for i, l in enumerate(second) if l == ["wait", event, "0x2000"]]
writes = [i for i, l in enumerate(second)
          if l[0] == "copy" or (l[0] == "launch" and "upload_table" in l[1])]
assert waits and writes and waits[0] < writes[0], second
if not small:
    assert second[writes[0]][2] != first[table[0]][2], (first, second)
assert run(S[1]) == 0
assert log()[0] == ["sync", event], log()
F.fake_clear_log()
L.svo_batch_destroy(b)
assert sum(l[0] == "sync" for l in log()) == 2, log()
""")


def test_an_error_left_by_another_call_is_not_a_launchs():
    """Any failed HIP call of the thread, the caller's own included, leaves its error
    for hipGetLastError; launches that succeed do not answer with it."""
    fakehip.run(PRELUDE + """
b = C.c_void_p()
assert L.svo_batch_create(4, C.byref(b)) == 0
js = jobs(render(), cast(BIG), cast(100))
hits = C.byref(N.Hits())
vpc = vp.to_c()
out = np.zeros(40 * 24, np.uint32)
calls = dict(
    batch=lambda: L.svo_batch_run(b, js, 3, S[0]),
    static=lambda: L.svo_batch_run_static(js, 3, S[0]),
    cast=lambda: L.svo_cast(tree._h, rays.ctypes.data, 100, hits, S[0]),
    stream=lambda: L.svo_cast(tree._h, rays.ctypes.data, BIG, hits, S[0]),
    lod=lambda: L.svo_cast_at_lod(tree._h, rays.ctypes.data, 100, 9.0, hits, S[0]),
    frame=lambda: L.svo_render(tree._h, C.byref(vpc), 40, 24, hits, S[0]),
    frame_lod=lambda: L.svo_render_at_lod(tree._h, C.byref(vpc), 40, 24, 9.0, hits, S[0]),
    shaded=lambda: L.svo_render_rgba8(tree._h, C.byref(vpc), 40, 24, 0, out.ctypes.data, S[0]))
F.fake_leave_error.restype = None
wrong = []
for name, call in calls.items():
    F.fake_leave_error()
    if call() != 0:
        wrong.append((name, error()))
    assert call() == 0
assert not wrong, wrong
# and a launch that fails still says so
for name, kernel in dict(batch="batch_tile", static="batch_tile", cast="cast_kernel",
                         stream="cast_stream", lod="cast_lod", frame="frame_kernel",
                         frame_lod="frame_lod", shaded="shade").items():
    F.fake_fail_launch(kernel.encode())
    assert calls[name]() == 7, name
    F.fake_fail_launch(b"")
L.svo_batch_destroy(b)
""")
