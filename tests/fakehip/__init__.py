"""Runs a function of this package's cases in a CPU process whose HIP runtime
is the stand-in of fakehip.cpp (tests only)."""
from __future__ import annotations

import os
import subprocess
import sys
from pathlib import Path

HERE = Path(__file__).resolve().parent
LIB = HERE / "libfakehip.so"
ROOT = HERE.parent.parent


def run(code: str) -> str:
    """Standard output of `code` in such a process; raises if it fails."""
    subprocess.run(["make", "-s", "-C", str(HERE)], check=True)
    env = dict(os.environ, PYTHONPATH=f"{ROOT}:{HERE.parent}",
               LD_PRELOAD=" ".join(filter(None, [str(LIB), os.environ.get("LD_PRELOAD")])))
    p = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True,
                       timeout=300)
    assert p.returncode == 0, f"exit code {p.returncode}\n{p.stdout}{p.stderr}"
    return p.stdout
