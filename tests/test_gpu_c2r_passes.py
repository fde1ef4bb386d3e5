"""The power-of-two c2r passes: the first pass of an even-length four-step c2r (bin pairs through
buffers, IO code 66, 82 for float bins), outputs stored as complex words where rows allow it and as
real words where they do not, and the Bluestein c2r of odd pairs (chirp-in and chirp-out instances).
Against the long-double oracle at the parity bars: 1e-12, and for float32 arrays 2^-24 (one rounding)
plus the FP64 error."""
import ctypes

import numpy as np
import pytest

import oracle
from impulse_amd import _lib, synth
from impulse_amd import fft as F
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu
TOL = {"f64": 1e-12, "f32": 2.0 ** -24 + 2e-15}


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


def _c2r(n, batch, dt, fwd, pitch, offset, kind=None, reverse=False):
    """c2r (or its r2c-adjoint kind) of [batch, n/2+1] random bins into rows `pitch` apart, `offset`
    elements into the buffer, or with the rows in reverse order; returns output, bins and kernels."""
    import torch
    h = synth.complex_normal((batch, n // 2 + 1), seed=n + batch)
    if dt == "f32":
        h = h.astype(np.complex64)
    hd = torch.from_numpy(h).cuda()
    buf = torch.zeros(offset + batch * pitch, dtype=torch.float32 if dt == "f32" else torch.float64, device="cuda")
    es = buf.element_size()
    st = -pitch * es if reverse else pitch * es
    base = buf.data_ptr() + offset * es + ((batch - 1) * pitch * es if reverse else 0)
    pl = F.Plan(_lib.C2R if kind is None else kind, [batch, n], [(n // 2 + 1) * 2 * es, 2 * es], [st, es], [1], fwd,
                dtype=_lib.F32 if dt == "f32" else _lib.F64)
    pl.execute(hd.data_ptr(), base, 0.25, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    rows = buf.cpu().numpy()[offset:].reshape(batch, pitch)
    assert not rows[:, n:].any() and not buf.cpu().numpy()[:offset].any()   # nothing beside the rows
    return (rows[::-1] if reverse else rows)[:, :n], h, _names(pl)


@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("n", [1 << 15, 1 << 17, 1 << 18, 1 << 21])
def test_four_step_even(n, dt):
    for batch, fwd, pitch, offset, rev in ((1, False, n, 0, False), (3, True, n + 2, 0, False), (2, False, n + 1, 0, False),
                                           (2, True, n, 1, False), (3, False, n + 2, 2, True)):
        y, h, names = _c2r(n, batch, dt, fwd, pitch, offset, reverse=rev)
        wide = h.astype(np.complex128)
        assert rel_l2(y, oracle.c2r(wide, n, [1], fwd, 0.25)) <= TOL[dt], (n, batch, fwd, pitch, offset)
        assert names[0].endswith(", 1, %d>" % (82 if dt == "f32" else 66)), names


@pytest.mark.parametrize("n", [1 << 12, 1 << 15, 1 << 17])
def test_adjoint_of_r2c(n):
    """<A x, y> = <x, A* y>: all bins but 0 and n/2 take half the weight."""
    gx, y, _ = _c2r(n, 2, "f64", True, n, 0, kind=_lib.R2C_ADJOINT)
    x = synth.uniform((2, n), -1.0, 1.0, seed=3)
    ax = oracle.r2c(x, [1], True, 0.25)
    lhs = float(np.sum(ax.real * y.real + ax.imag * y.imag))
    assert abs(lhs - float(np.sum(x * gx))) <= 1e-12 * np.linalg.norm(ax) * np.linalg.norm(y)


@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("n,batch", [(32749, 1), (32749, 4), (60013, 3)])
def test_bluestein_odd_pairs(n, batch, dt):
    for fwd in (False, True):
        y, h, names = _c2r(n, batch, dt, fwd, n, 0)
        assert rel_l2(y, oracle.c2r(h.astype(np.complex128), n, [1], fwd, 0.25)) <= TOL[dt], (n, batch, fwd)
        codes = [int(s.rsplit(",", 1)[1].rstrip(">")) for s in names]
        base = [c & 7 for c in codes]
        assert base == [5, 4, 6], names
