import json
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) GPU")


@pytest.fixture(scope="session")
def golden():
    import numpy as np
    return np.load(os.path.join(ROOT, "tests", "golden", "golden.npz"))


def rel_l2(a, b):
    import numpy as np
    a = np.asarray(a)
    b = np.asarray(b)
    den = np.linalg.norm(b)
    return float(np.linalg.norm(a - b) / (den if den > 0 else 1.0))


_STAND_IN = os.path.join(ROOT, "tests", "cpp", "hip_stand_in.cpp")
_HOST_PRELUDE = """
import ctypes, json, sys
S = ctypes.CDLL({so!r}, mode=ctypes.RTLD_GLOBAL)
S.standin_launches.restype = ctypes.c_char_p
S.standin_limit.argtypes = [ctypes.c_size_t]
S.standin_used.restype = S.standin_peak.restype = ctypes.c_size_t
sys.path.insert(0, {root!r})
from impulse_amd import _lib
L = _lib.lib()
def launches():
    return [l.split() for l in S.standin_launches().decode().splitlines()]
def report(x):
    print("REPORT " + json.dumps(x))
"""


@pytest.fixture(scope="session")
def hip_host(tmp_path_factory):
    """Runs a snippet in a process whose HIP runtime is the stand-in of tests/cpp/hip_stand_in.cpp and
    returns what it passed to report().  The snippet finds L (the library), _lib, S (the stand-in's
    switches) and launches() (name, grid x, grid y, block, LDS bytes of every launch since the last call)."""
    so = str(tmp_path_factory.mktemp("standin") / "hip_stand_in.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-std=c++17", "-I/opt/rocm/include", _STAND_IN, "-o", so],
                   check=True)

    def run(code, timeout=120):
        r = subprocess.run([sys.executable, "-c", _HOST_PRELUDE.format(so=so, root=ROOT) + code],
                           capture_output=True, text=True, timeout=timeout)
        assert r.returncode == 0, (r.returncode, r.stdout[-2000:], r.stderr[-2000:])
        last = [l for l in r.stdout.splitlines() if l.startswith("REPORT ")]
        assert last, r.stdout
        return json.loads(last[-1][len("REPORT "):])

    run.so = so
    return run
