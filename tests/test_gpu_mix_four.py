"""Real four-step transforms of smooth lengths that are no power of two: their first and last passes on the
mixed-radix kernel (real words and odd pairs into twiddled columns, rows stored as real words), with aligned rows, odd pitches and offsets, rows in reverse order, float arrays and the adjoint kinds.
Against the long-double oracle at the parity bars: 1e-12, and for float32 arrays 2^-24 (one rounding) plus the
FP64 error."""
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


def _rows(a, pitch, offset, reverse):
    """`a`'s rows on the device, `pitch` elements apart from element `offset` on (the last row first when
    `reverse`): buffer, address of row 0, row stride in bytes."""
    import torch
    es = a.dtype.itemsize
    buf = np.zeros(offset + len(a) * pitch, dtype=a.dtype)
    v = buf[offset:].reshape(len(a), pitch)
    v[:, :a.shape[1]] = a[::-1] if reverse else a
    d = torch.from_numpy(buf).cuda()
    st = -pitch * es if reverse else pitch * es
    return d, d.data_ptr() + offset * es + ((len(a) - 1) * pitch * es if reverse else 0), st


@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("kind,adj", [("r2c", 0), ("c2r", 0), ("r2c", 1), ("c2r", 1)])
@pytest.mark.parametrize("n,batch,extra,offset,reverse", [
    (18000, 1, 0, 0, False), (48000, 3, 0, 0, False), (44100, 2, 1, 1, False), (22022, 2, 2, 0, True),
    (9009, 3, 0, 0, False), (30375, 2, 1, 1, True), (11025, 1, 0, 0, False)])
def test_real_four_step(n, batch, extra, offset, reverse, kind, adj, dt):
    """kind r2c with adj: the adjoint of c2r (interior bins doubled); c2r with adj: the adjoint of r2c (halved)."""
    import torch
    print(f"case {kind} adj={adj} {batch} x {n} extra={extra} offset={offset} reverse={reverse} {dt}", flush=True)
    h = n // 2 + 1
    r = synth.uniform((batch, n), -1, 1, seed=n)
    c = synth.complex_normal((batch, h), seed=n + 1)
    if dt == "f32":
        r, c = r.astype(np.float32), c.astype(np.complex64)
    rd, rp, rs = _rows(r if kind == "r2c" else np.zeros_like(r), n + extra, offset, reverse)
    cd, cp, cs = _rows(c if kind == "c2r" else np.zeros_like(c), h + extra, offset, reverse)
    weights = np.ones(h)
    weights[1:(n - 1) // 2 + 1] = 2.0
    for fwd in (True, False):
        if kind == "r2c":
            code, src, dst = (_lib.C2R_ADJOINT if adj else _lib.R2C), rp, cp
            ist, ost = [rs, r.itemsize], [cs, c.itemsize]
            want = oracle.r2c(r.astype(np.float64), [1], not fwd if adj else fwd, 0.25) * (weights if adj else 1.0)
        else:
            code, src, dst = (_lib.R2C_ADJOINT if adj else _lib.C2R), cp, rp
            ist, ost = [cs, c.itemsize], [rs, r.itemsize]
            want = oracle.c2r(c.astype(np.complex128) / (weights if adj else 1.0), n, [1], not fwd if adj else fwd, 0.25)
        pl = F.Plan(code, [batch, n], ist, ost, [1], fwd, dtype=_lib.F32 if dt == "f32" else _lib.F64)
        pl.execute(src, dst, 0.25, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        buf = (cd if kind == "r2c" else rd).cpu().numpy()
        m = h if kind == "r2c" else n
        rows = buf[offset:].reshape(batch, m + extra)
        assert not buf[:offset].any() and not rows[:, m:].any()   # nothing beside the rows
        got = (rows[::-1] if reverse else rows)[:, :m]
        assert rel_l2(got, want) < TOL[dt], (kind, fwd)
        names = _names(pl)
        print(names, flush=True)
        # the columns of half-spectrum bins stay on the generic kernel
        assert sum(s.startswith("k_fft_mix") for s in names) == (2 if kind == "r2c" else 1), names
