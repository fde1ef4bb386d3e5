"""Planning on the host (no GPU): the stand-in HIP runtime of tests/cpp/hip_stand_in.cpp."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PLAN = """
import time
def strides(shape, e):
    st = [e]
    for n in reversed(shape[1:]):
        st.insert(0, st[0] * n)
    return _lib.strides(st)
def plan(kind, dtype, shape, axes):
    half = list(shape)
    half[axes[-1]] = shape[axes[-1]] // 2 + 1
    e = 4 if dtype else 8
    h = ctypes.c_void_p()
    rc = L.impulse_fft_plan_create(ctypes.byref(h), kind, dtype, len(shape), _lib.sizes(shape),
                                   strides(half if kind == 2 else shape, e if kind == 1 else 2 * e),
                                   strides(half if kind == 1 else shape, e if kind == 2 else 2 * e),
                                   len(axes), _lib.sizes(axes), 1)
    assert rc == 0, L.impulse_fft_last_error()
    return h
"""


@pytest.mark.parametrize("n", [1999, 3851])
def test_bluestein_length_is_searched_once(hip_host, n):
    # The candidate lengths of a Bluestein axis are factored once, in microseconds each: such a plan
    # takes little more than its tables, not several searches.  It computes about four tables of its
    # padded length (4,000 and 8,192 points); the plan of 8,192 points, with one such table, is the measure.
    mine, measure = hip_host(PLAN + f"""
best = [1.0, 1.0]
for _ in range(9):
    for k, m in enumerate(({n}, 8192)):
        t = time.process_time()
        h = plan(0, 0, [1, m], [1])
        best[k] = min(best[k], time.process_time() - t)
        L.impulse_fft_plan_destroy(h)
report(best)
""")
    assert mine < (4.5 if n < 2000 else 8) * measure


def test_four_step_keeps_the_tables_it_reads(hip_host):
    # A smooth four-step pass on the mixed-radix kernel reads stage tables only: the plan holds the two
    # levels of W_n (two times about sqrt(n) entries), the stage tables of both factors (fewer entries
    # than points) and two workspaces.
    n, l1, l2 = 300000, 600, 500
    held = hip_host(PLAN + f"report(L.impulse_fft_plan_device_bytes(plan(0, 0, [1, {n}], [1])))")
    s = 1
    while s * s < n:
        s *= 2
    assert held <= 16 * (2 * n + s + (n + s - 1) // s + 1 + l1 + l2)


def test_long_bluestein_keeps_one_spectrum(hip_host):
    # The three-pass Bluestein reads its kernel's spectrum in row order: that table alone is kept.
    n, n2 = 100003, 262144
    held = hip_host(PLAN + f"report(L.impulse_fft_plan_device_bytes(plan(0, 0, [1, {n}], [1])))")
    assert held <= 16 * (2 * n2 + n + 2048)   # workspace, spectrum, chirp, the tables of 512-point passes


def test_small_workgroups_keep_their_mode(hip_host, tmp_path):
    """The spectrum product and the row pairs are not in the per-point path of the power-of-two kernel: its
    small workgroups run them on an instance of their own, or refuse, on any grid."""
    exe = str(tmp_path / "pow2_small")
    lib = os.path.join(ROOT, "impulse_amd")
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I", os.path.join(lib, "csrc"), os.path.join(ROOT, "tests", "cpp", "pow2_small_main.cpp"),
                    "-o", exe, hip_host.so, "-L", lib, "-l:libimpulse_fft.so", f"-Wl,-rpath,{lib}",
                    f"-Wl,-rpath,{os.path.dirname(hip_host.so)}", "-Wl,--allow-shlib-undefined"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    lines = [l.split() for l in r.stdout.splitlines()]
    assert len(lines) == 12
    for conv, mode, grid, err, name, *_ in lines:
        if conv == "1" and mode == "0":
            assert err == "0" and "k_fft_pow2ILi512ELi0ELi12ELi2E" in name, (grid, name)   # spectrum product, four-wave name
        else:
            assert err != "0" and name == "-", (conv, mode, grid, name)


def test_bluestein_lengths_find_their_kernel(hip_host):
    """Every non-smooth length whose padded transform fits one pass runs on the mixed-radix Bluestein kernel,
    also where many smooth lengths just above it need more threads than that kernel has."""
    got = hip_host(PLAN + """
got = {}
for n in list(range(17, 4096, 97)) + [3841, 3850, 3851, 3889, 3899, 3900, 3907, 4093, 4096]:
    h = plan(0, 0, [2, n], [1])
    L.impulse_fft_execute(h, 1 << 30, 1 << 31, 1.0, None)
    launches()
    L.impulse_fft_execute(h, 1 << 30, 1 << 31, 1.0, None)
    got[n] = [l[0] for l in launches()]
    L.impulse_fft_plan_destroy(h)
report(got)
""")
    for n, names in got.items():
        m = int(n)
        for p in (2, 3, 5, 7, 11, 13):
            while m % p == 0:
                m //= p
        if m > 1:
            assert len(names) == 1 and "k_fft_mix_blue" in names[0], (n, names)
