"""ctypes front end of libdevmath.so (tests only; see devmath.hip)."""
from __future__ import annotations

import ctypes as C
import subprocess
from pathlib import Path

HERE = Path(__file__).resolve().parent
LIB = HERE / "libdevmath.so"
_lib = None


def run(op: str, b, a=None):
    """"rcp" 1 / b, "quot" a / b or "sqrt" of a contiguous f32 device tensor."""
    global _lib
    import torch
    if _lib is None:
        if not LIB.exists():
            subprocess.run(["make", "-s", "-C", str(HERE)], check=True)
        _lib = C.CDLL(str(LIB))
        _lib.devmath.argtypes = [C.c_int, C.c_void_p, C.c_void_p, C.c_void_p, C.c_uint32,
                                 C.c_void_p]
    for t in (b,) if a is None else (a, b):
        assert t.dtype == torch.float32 and t.is_contiguous() and t.shape == b.shape
    out = torch.empty_like(b)
    st = _lib.devmath(("rcp", "quot", "sqrt").index(op), None if a is None else a.data_ptr(),
                      b.data_ptr(), out.data_ptr(), b.numel(),
                      torch.cuda.current_stream().cuda_stream)
    assert st == 0, st
    return out
