"""The GPU tests' lengths against the factoring the library gives all lengths of the mixed-radix kernel (no
GPU: the stand-in HIP runtime of tests/cpp/hip_stand_in.cpp)."""
import os
import subprocess

from tests.conftest import ROOT
from tests.mix_lengths import LENGTHS


def _places(radices):
    last = len(radices) - 1
    return {("first" if k == 0 else "last" if k == last else "between", r) for k, r in enumerate(radices)} | {
        ("stages", len(radices))}


def test_lengths_cover_the_factoring(hip_host, tmp_path):
    exe, lib = str(tmp_path / "mix_factor"), os.path.join(ROOT, "impulse_amd")
    subprocess.run(["g++", "-O1", "-std=c++17", os.path.join(ROOT, "tests", "cpp", "mix_factor_main.cpp"), "-o", exe,
                    hip_host.so, "-L", lib, "-l:libimpulse_fft.so", f"-Wl,-rpath,{lib}",
                    f"-Wl,-rpath,{os.path.dirname(hip_host.so)}", "-Wl,--allow-shlib-undefined"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, check=True)
    got = {v[0]: v[1:] for v in ([int(w) for w in l.split()] for l in r.stdout.splitlines())}
    assert len(got) > 500
    for n, radices in got.items():
        p = 1
        for x in radices:
            p *= x
        assert p == n and 2 <= len(radices) <= 6
    want = set().union(*(_places(v) for v in got.values()))
    assert set().union(*(_places(got[n]) for n in LENGTHS)) == want
