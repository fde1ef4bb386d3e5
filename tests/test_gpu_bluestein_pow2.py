"""Long Bluestein transforms on the next power of two, far above the smallest smooth length or next to it:
three passes in every kind, batches whose workspace passes 2 GiB in chunks, and the plans that keep the smooth
length because only that fits the scratch of execution without allocation.  Against the long-double oracle at
the parity bar of 1e-12."""
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


def _plan(kind, batch, n, fwd):
    import torch
    if kind == "r2c":
        x = synth.uniform((batch, n), -1, 1, seed=n + batch)
    else:
        x = synth.complex_normal((batch, n // 2 + 1 if kind == "c2r" else n), seed=n + batch)
    xd = torch.from_numpy(x).cuda()
    shape, dt = (batch, n // 2 + 1 if kind == "r2c" else n), torch.float64 if kind == "c2r" else torch.complex128
    yd = torch.empty(shape, dtype=dt, device="cuda")
    pl = F.Plan({"c2c": _lib.C2C, "r2c": _lib.R2C, "c2r": _lib.C2R}[kind], [batch, n],
                [s * xd.element_size() for s in xd.stride()], [s * yd.element_size() for s in yd.stride()], [1], fwd)
    return x, xd, yd, pl


def _want(kind, row, n, fwd):
    if kind == "c2r":
        return oracle.c2r(row, n, [0], fwd, 0.5)
    return (oracle.c2c if kind == "c2c" else oracle.r2c)(row, [0], fwd, 0.5)


# 4,099 and 131,101: power of two 1.99 times the smooth length; 100,003: 1.31; 65,521: 1.0 below 2^17;
# 262,202 = 2 * 131,101: even real lengths run on half of it
@pytest.mark.parametrize("kind,batch,n", [
    ("c2c", 1, 4099), ("c2c", 70, 4099), ("c2c", 3, 100003), ("c2c", 2, 65521), ("r2c", 5, 4099), ("r2c", 3, 100003),
    ("r2c", 2, 262202), ("c2r", 5, 4099), ("c2r", 3, 131101), ("c2r", 2, 262202), ("c2c", 1, 1048583)])
@pytest.mark.parametrize("fwd", [True, False])
def test_three_passes(kind, batch, n, fwd):
    import torch
    print(f"case {kind} {batch} x {n} fwd={fwd}", flush=True)
    x, xd, yd, pl = _plan(kind, batch, n, fwd)
    pl.execute(xd.data_ptr(), yd.data_ptr(), 0.5, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    y = yd.cpu().numpy()
    for row in {0, batch - 1}:
        assert rel_l2(y[row], _want(kind, x[row], n, fwd)) < TOL, (kind, batch, n, row)
    names = _names(pl)
    assert len(names) == (4 if kind == "r2c" else 3) and all(s.startswith(("k_fft_pow2", "k_real_post")) for s in names)


def test_batch_past_two_gib():
    """c2c of 1,100 x 100,003: 4.6 GB of workspace in chunks of 511 signals."""
    import torch
    batch, n = 1100, 100003
    print(f"case chunks {batch} x {n}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(3)
    xd = torch.view_as_complex(torch.randn((batch, n, 2), dtype=torch.float64, device="cuda", generator=g))
    yd = torch.empty_like(xd)
    st = [n * 16, 16]
    pl = F.Plan(_lib.C2C, [batch, n], st, st, [1], True)
    pl.execute(xd.data_ptr(), yd.data_ptr(), 0.5, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert len(_names(pl)) == 9
    for row in (0, 510, 511, 1021, 1022, 1099):
        assert rel_l2(yd[row].cpu().numpy(), _want("c2c", xd[row].cpu().numpy(), n, True)) < TOL, row


@pytest.mark.parametrize("kind,batch,smooth", [("r2c", 12, False), ("r2c", 14, True), ("c2c", 7, False),
                                               ("c2r", 14, False)])
def test_scratch_limit(kind, batch, smooth):
    """131,101 points: every plan whose smooth length's two workspace arrays fit 64 MiB still runs without
    allocation; r2c of 14 rows fits only with the smooth length, and keeps it."""
    import torch
    n = 131101
    print(f"case scratch {kind} {batch} x {n}", flush=True)
    x, xd, yd, pl = _plan(kind, batch, n, True)
    zd = torch.empty_like(yd)
    s = torch.cuda.current_stream().cuda_stream
    pl.execute(xd.data_ptr(), yd.data_ptr(), 0.5, s)
    _lib.check(_lib.lib().impulse_fft_execute_noalloc(pl.handle, xd.data_ptr(), zd.data_ptr(), 0.5, s))
    torch.cuda.synchronize()
    assert torch.equal(torch.view_as_real(yd) if yd.is_complex() else yd, torch.view_as_real(zd) if zd.is_complex() else zd)
    assert rel_l2(zd[batch - 1].cpu().numpy(), _want(kind, x[batch - 1], n, True)) < TOL
    assert any(v.startswith(("k_fft_lds", "k_fft_mix")) for v in _names(pl)) == smooth
