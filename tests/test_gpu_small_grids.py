"""Power-of-two passes of 128 to 1,024 points on grids too small for the chip, which take fewer transforms
per workgroup: rows, columns, four-step passes and three-pass Bluestein, and the per-point instances that
real axes and odd row pitches need.  Against the long-double oracle at the parity bar of 1e-12."""
import ctypes

import numpy as np
import pytest

import oracle
from impulse_amd import _lib, synth
from impulse_amd import fft as F
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu
TOL = 1e-12


@pytest.fixture(scope="module", autouse=True)
def _device():
    import torch   # before the library: both then share one HIP runtime
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    yield
    torch.cuda.synchronize()


def _names(plan):
    out = []
    for k in range(plan.num_launches):
        name = ctypes.create_string_buffer(64)
        z, u = ctypes.c_size_t(), ctypes.c_uint()
        _lib.check(_lib.lib().impulse_fft_plan_pass_info(plan.handle, k, name, 64, ctypes.byref(z), ctypes.byref(z),
                                                      ctypes.byref(u), ctypes.byref(u), ctypes.byref(z)))
        out.append(name.value.decode())
    return out


def _run(kind, shape, axis, pad, fwd):
    """One transform along `axis` of a C-ordered array whose output's rows are `pad` elements longer than
    they need; returns the output, the oracle's and the kernels that ran."""
    import torch
    half = list(shape)
    half[axis] = shape[axis] // 2 + 1
    ish = half if kind == "c2r" else list(shape)
    osh = half if kind == "r2c" else list(shape)
    seed = sum(shape)
    x = synth.uniform(tuple(ish), -1, 1, seed=seed) if kind == "r2c" else synth.complex_normal(tuple(ish), seed=seed)
    xd = torch.from_numpy(x).cuda()
    yd = torch.full([osh[0], osh[1] + pad], 7.0, dtype=torch.float64 if kind == "c2r" else torch.complex128,
                    device="cuda")
    pl = F.Plan({"c2c": _lib.C2C, "r2c": _lib.R2C, "c2r": _lib.C2R}[kind], shape,
                [s * xd.element_size() for s in xd.stride()], [s * yd.element_size() for s in yd.stride()],
                [axis], fwd)
    pl.execute(xd.data_ptr(), yd.data_ptr(), 0.5, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    y = yd.cpu().numpy()
    assert (y[:, osh[1]:] == 7.0).all()   # nothing beside the rows
    if kind == "c2r":
        want = oracle.c2r(x, shape[axis], [axis], fwd, 0.5)
    else:
        want = (oracle.c2c if kind == "c2c" else oracle.r2c)(x, [axis], fwd, 0.5)
    return y[:, :osh[1]], want, _names(pl)


@pytest.mark.parametrize("fwd", [True, False])
@pytest.mark.parametrize("kind,shape,axis,pad,small", [
    # rows: one, a ragged last workgroup, the last small grid (255 full workgroups) and the first full one
    ("c2c", [1, 128], 1, 0, 1), ("c2c", [13, 256], 1, 0, 1), ("c2c", [3, 512], 1, 0, 1), ("c2c", [5, 1024], 1, 1, 1),
    ("c2c", [4080, 256], 1, 0, 1), ("c2c", [4081, 256], 1, 0, 0),
    ("r2c", [7, 256], 1, 0, 1), ("r2c", [3, 2048], 1, 0, 1), ("c2r", [9, 512], 1, 0, 1), ("c2r", [2, 2048], 1, 3, 1),
    # columns
    ("c2c", [128, 13], 0, 0, 1), ("c2c", [256, 5], 0, 2, 1), ("c2c", [512, 3], 0, 0, 1), ("c2c", [1024, 9], 0, 0, 1),
    ("r2c", [1024, 5], 0, 0, 0), ("c2r", [1024, 5], 0, 0, 1),
    # four-step: 128 x 128, 256 x 128, 512 x 256, 1024 x 1024; odd row pitches take the per-point stores
    ("c2c", [1, 16384], 1, 0, 2), ("c2c", [3, 32768], 1, 1, 2), ("c2c", [1, 131072], 1, 0, 2),
    ("r2c", [1, 32768], 1, 0, 2), ("r2c", [2, 262144], 1, 0, 2),
    ("c2r", [1, 32768], 1, 0, 2), ("c2r", [3, 65536], 1, 1, 2), ("c2r", [1, 524288], 1, 0, 2),
    # Bluestein, three passes
    ("c2c", [1, 8191], 1, 0, 3), ("c2c", [3, 30011], 1, 0, 3), ("r2c", [1, 8191], 1, 0, 3),
    ("r2c", [3, 60013], 1, 0, 3), ("c2r", [3, 8191], 1, 0, 3), ("c2r", [2, 16382], 1, 0, 3)])
def test_small_grids(kind, shape, axis, pad, small, fwd):
    print(f"case {kind} {shape} axis={axis} pad={pad} fwd={fwd}", flush=True)
    y, want, names = _run(kind, shape, axis, pad, fwd)
    print(names, flush=True)
    assert rel_l2(y, want) < TOL
    assert sum("_tb" in s for s in names) >= small, names
    if not small:
        assert not any("_tb" in s for s in names), names
