"""The rules by which calls are addressed and dispatched, on the CPU: compiles
tests/native/launch_rules.cpp (host side only) against the library's own headers
and runs its checks. What the kernels do with a wrong rule would be a read out
of range or a slower kernel, which no comparison of outputs shows.
"""
from __future__ import annotations

import subprocess
import sys
from pathlib import Path

NATIVE = Path(__file__).resolve().parent / "native"


def test_launch_rules():
    sys.path.insert(0, str(NATIVE))
    try:
        import build
    finally:
        sys.path.remove(str(NATIVE))
    result = subprocess.run([str(build.build_launch_rules())], capture_output=True, text=True, timeout=120)
    assert result.returncode == 0 and "launch rules OK" in result.stdout, result.stdout + result.stderr
