"""Runs a script against libportlbm_hip.so on the CPU, with the HIP runtime of
tests/cpp/hip_stand_in.cpp in place of libamdhip64 (a process of its own: the
stand-in has to be loaded before the library).

In the script: `pa` is the package, `fail(entry_point, nth_call)`,
`memory(bytes)`, `log()` (kernels launched since the last call, by name) and
`live()` (device bytes, host bytes, handles) control and watch the stand-in;
`log` fails where the library touched what it should not.
"""
import os
import shutil
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
HIP_INCLUDE = Path(os.environ.get("ROCM_PATH", "/opt/rocm")) / "include"

PRELUDE = f"""
import ctypes, sys
s = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path.insert(0, {str(ROOT)!r})
import numpy as np
import portlbm_amd as pa
s.stand_in_log.restype = ctypes.c_char_p
def fail(what, after):
    s.stand_in_fail(what.encode(), after)
def memory(n):
    s.stand_in_memory(ctypes.c_size_t(n))
def log():
    lines = s.stand_in_log().decode().splitlines()
    assert not [l for l in lines if l.startswith("BAD")], lines
    return [l.removeprefix("launch ") for l in lines]
def live():
    out = (ctypes.c_size_t * 3)()
    s.stand_in_live(out)
    return list(out)
def raises(f):
    try:
        f()
    except pa.LbmError as e:
        return str(e)
    raise AssertionError("was not refused")
"""


def build(directory: Path) -> Path:
    if shutil.which("g++") is None or not (HIP_INCLUDE / "hip" / "hip_runtime_api.h").exists():
        pytest.skip("needs g++ and the HIP headers")
    so = directory / "hip_stand_in.so"
    subprocess.run(["g++", "-std=c++20", "-O1", "-g", "-shared", "-fPIC", "-pthread", f"-I{HIP_INCLUDE}",
                    str(ROOT / "tests" / "cpp" / "hip_stand_in.cpp"), "-o", str(so)], check=True)
    return so


def run(so: Path, script: str) -> None:
    r = subprocess.run([sys.executable, "-c", PRELUDE + script, str(so)], stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-4000:]
