"""Host side of the DCT / DST plans (no GPU): the route of an axis and how far a workgroup's lines reach.
The HIP runtime is the stand-in of tests/cpp/hip_stand_in.cpp."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_line_reach(tmp_path):
    """line_reach holds the offsets of every group, over packed, padded, broadcast and reversed arrays."""
    exe = str(tmp_path / "line_reach")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "impulse_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "line_reach_main.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0 and int(r.stdout) == 40000, r.stdout


# arrays of 2.1 to 8.4 GB; the lines of the last two are longer than 31-bit offsets
@pytest.mark.parametrize("shape,strides,axis,launches", [
    ((33000, 8192), None, 1, 1),
    ((3, 1500001, 64), (1500001 * 65, 65, 1), 2, 1),
    ((33000, 8192), (-8192, 1), 1, 1),
    ((5, 1024, 60000), None, 1, 1),
    ((270000, 1000), (1000, 1), 0, None),
    ((2, 1000), (1 << 29, 1 << 19), 1, None),
])
def test_arrays_over_2_gib_keep_one_kernel(hip_host, shape, strides, axis, launches):
    if strides is None:
        strides, acc = [], 1
        for n in reversed(shape):
            strides.insert(0, acc)
            acc *= n
    got = hip_host(f"""
shape, st, got = {list(shape)}, _lib.strides([8 * s for s in {list(strides)}]), []
for t in (2, 3, 4):
    h = ctypes.c_void_p()
    rc = L.impulse_fft_r2r_plan_create(ctypes.byref(h), 5, t, 0, 0, len(shape), _lib.sizes(shape), st, st, 1,
                                       _lib.sizes([{axis}]))
    assert rc == 0, L.impulse_fft_last_error()
    got.append(L.impulse_fft_plan_num_launches(h))
    L.impulse_fft_plan_destroy(h)
report(got)
""")
    if launches is None:
        assert min(got) > 1
    else:
        assert got == [launches] * 3


@pytest.mark.parametrize("shape,axis", [((2000, 30), 1), ((300, 16), 1), ((2000, 10), 1), ((200000, 30), 1), ((20000, 16), 1),
                                        ((2000, 90), 1), ((128, 2000), 0), ((30, 2000), 0), ((64, 300), 0)])
def test_short_lines_fill_wavefronts(hip_host, shape, axis):
    """Many short lines: no workgroup under a wavefront, and several threads a line along rows."""
    got = hip_host(f"""
shape, got = {list(shape)}, []
st = _lib.strides([8 * shape[1], 8])
for t in (2, 3, 4):
    h = ctypes.c_void_p()
    rc = L.impulse_fft_r2r_plan_create(ctypes.byref(h), 5, t, 0, 0, 2, _lib.sizes(shape), st, st, 1, _lib.sizes([{axis}]))
    assert rc == 0, L.impulse_fft_last_error()
    launches()
    assert L.impulse_fft_execute(h, 1 << 30, 1 << 32, 1.0, None) == 0
    got += launches()
report(got)
""")
    assert len(got) == 3 and all("k_r2r_mix" in l[0] for l in got)
    lines = shape[1 - axis]
    for _, grid, _, block, _ in got:
        assert int(block) >= 64
        if axis == 1:
            assert int(block) * int(grid) >= 2 * lines


@pytest.mark.parametrize("n,threads", [(16, 4), (90, 32), (2048, 512), (6250, 512)])
def test_single_line_uses_more_threads(hip_host, n, threads):
    """One line alone is bound by a thread's chain: a thread for every two points, up to 512."""
    got = hip_host(f"""
h, st = ctypes.c_void_p(), _lib.strides([8 * {n}, 8])
assert L.impulse_fft_r2r_plan_create(ctypes.byref(h), 5, 2, 0, 0, 2, _lib.sizes([1, {n}]), st, st, 1, _lib.sizes([1])) == 0
launches()
assert L.impulse_fft_execute(h, 1 << 30, 1 << 32, 1.0, None) == 0
report(launches())
""")
    assert len(got) == 1 and int(got[0][3]) == threads
