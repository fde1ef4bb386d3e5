"""GPU parity of the mixed-radix pass kernel (fft_mix.hip): lengths of two, three and four stages,
every radix 2..16 as first, middle and last stage, partial workgroups, both lane mappings, strided
and reversed views, both precisions and the adjoint weights, against the long-double oracle.

Bars: 1e-12 relative L2 for float64 arrays (as every parity test of the engine); for float32 arrays
each output is the FP64 result rounded once, so 2^-24 of its magnitude plus the FP64 error.
"""
import ctypes

import numpy as np
import pytest

import oracle
from impulse_amd import _lib, synth
from impulse_amd import fft as F
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu
TOL = {"f64": 1e-12, "f32": 2.0 ** -24 + 2e-15}

# 17..26: the shortest lengths it takes (two stages); 169 = 13^2, 2197 = 13^3, 121, 1331: one prime in
# every stage; 200 (first stage 5, 8 ...), 360 .. 1920: composite radices; 4095, 4290: four stages of
# mixed primes; 5000, 6000: the longest four-stage lengths within a workgroup's threads
LENGTHS = [18, 20, 21, 24, 26, 33, 36, 91, 96, 120, 121, 125, 143, 169, 200, 231, 360, 405, 500, 686, 960, 1001,
           1080, 1331, 1536, 1920, 2197, 2250, 3003, 3072, 4095, 4290, 5000, 6000]


@pytest.fixture(scope="module", autouse=True)
def _device():
    import torch   # before the library: both then share one HIP runtime
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    yield
    torch.cuda.synchronize()


def _rand(shape, cplx, dt, seed):
    x = synth.complex_normal(shape, seed=seed) if cplx else synth.uniform(shape, -1.0, 1.0, seed=seed)
    if dt == "f32":
        x = x.astype(np.complex64 if cplx else np.float32)
    return x


def _wide(x):
    return x.astype(np.complex128 if np.iscomplexobj(x) else np.float64)


def _kernels(plan):
    out = []
    for k in range(plan.num_launches):
        name = ctypes.create_string_buffer(64)
        z, u = ctypes.c_size_t(), ctypes.c_uint()
        _lib.check(_lib.lib().impulse_fft_plan_pass_info(plan.handle, k, name, 64, ctypes.byref(z), ctypes.byref(z),
                                                      ctypes.byref(u), ctypes.byref(u), ctypes.byref(z)))
        out.append(name.value.decode())
    return out


def _run(kind, x, oshape, odt, axes, fwd, fct, n=None):
    """One device plan over C-contiguous arrays; returns the output and the kernels that ran."""
    import torch
    xd = torch.from_numpy(x).cuda()
    yd = torch.zeros(oshape, dtype=odt, device="cuda")
    shape = list(oshape) if kind == _lib.C2R else list(x.shape)
    st = [[s * t.element_size() for s in t.stride()] for t in (xd, yd)]
    f32 = x.dtype in (np.float32, np.complex64)
    pl = F.Plan(kind, shape, st[0], st[1], axes, fwd, dtype=_lib.F32 if f32 else _lib.F64)
    pl.execute(xd.data_ptr(), yd.data_ptr(), fct, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return yd.cpu().numpy(), _kernels(pl)


@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("n", LENGTHS)
def test_lengths(n, dt):
    """c2c of length n, r2c and c2r of lengths 2 n (half-length) and n (pairs where n is odd), rows and
    columns, with batches that leave the last workgroup partly filled."""
    import torch
    cdt, rdt = (torch.complex64, torch.float32) if dt == "f32" else (torch.complex128, torch.float64)
    for batch in (1, 7):
        for axis in (0, 1):
            shape = (n, batch) if axis == 0 else (batch, n)
            x = _rand(shape, True, dt, n + batch)
            for fwd in (True, False):
                y, ker = _run(_lib.C2C, x, shape, cdt, [axis], fwd, 0.5)
                assert all(k.startswith("k_fft_mix") for k in ker), (n, axis, ker)
                assert rel_l2(y, oracle.c2c(_wide(x), [axis], fwd, 0.5)) <= TOL[dt], (n, batch, axis, fwd)
            for m in ((n, 2 * n) if n % 2 else (2 * n,)):
                shape = (m, batch) if axis == 0 else (batch, m)
                half = [v // 2 + 1 if a == axis else v for a, v in enumerate(shape)]
                x = _rand(shape, False, dt, m + batch)
                y, ker = _run(_lib.R2C, x, half, cdt, [axis], True, 1.0)
                assert all(k.startswith("k_fft_mix") for k in ker), (m, axis, ker)
                assert rel_l2(y, oracle.r2c(_wide(x), [axis], True, 1.0)) <= TOL[dt], (m, batch, axis)
                h = _rand(tuple(half), True, dt, m)
                z, ker = _run(_lib.C2R, h, shape, rdt, [axis], False, 1.0 / m)
                assert all(k.startswith("k_fft_mix") for k in ker), (m, axis, ker)
                assert rel_l2(z, oracle.c2r(_wide(h), m, [axis], False, 1.0 / m)) <= TOL[dt], (m, batch, axis)


@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("n", [90, 105, 420])
def test_views(n, dt):
    """Strided and reversed axes, odd row pitches (real rows that are not aligned to complex words), an
    axis between two batch dimensions, both directions, in place."""
    cplx, real = _rand((3, 2 * n, 10), True, dt, 1), _rand((5, 2 * n + 1), False, dt, 2)
    tol = TOL[dt]
    for v in (cplx[:, ::2, :], cplx[::-1, n - 1::-1, ::3], cplx[:, ::-2, 1:8]):
        for fwd in (True, False):
            assert rel_l2(F.c2c(v, [1], fwd, 0.25), oracle.c2c(_wide(v), [1], fwd, 0.25)) <= tol
    buf = cplx[:, :n, :].copy()
    ref = oracle.c2c(_wide(buf), [1, 0], True, 1.0)
    F.c2c(buf, [1, 0], True, 1.0, out=buf)
    assert rel_l2(buf, ref) <= tol
    for v in (real[:, :n], real[:, 1:n + 1], real[::-1, n::-1][:, :n], real[:, ::2][:, :n]):
        for fwd in (True, False):
            assert rel_l2(F.r2c(v, [1], fwd, 1.0), oracle.r2c(_wide(v), [1], fwd, 1.0)) <= tol
    h = _rand((4, n, 7), True, dt, 3)
    for v, ax in ((h, 1), (h[:, ::-1, ::2], 1), (np.ascontiguousarray(h[0]).T, 1)):
        for fwd in (True, False):
            m = 2 * (v.shape[ax] - 1)
            for m in (m, m + 1):
                out = np.zeros([m if a == ax else s for a, s in enumerate(v.shape)] + [2],
                               np.float32 if dt == "f32" else np.float64)[..., 0]
                got = F.c2r(v, m, [ax], fwd, 1.0 / m, out=out)
                assert rel_l2(got, oracle.c2r(_wide(v), m, [ax], fwd, 1.0 / m)) <= tol, (m, ax, fwd)


@pytest.mark.parametrize("n", [90, 105, 1080])
def test_adjoint_weights(n):
    """<A x, y> = <x, A* y> of both real transforms over rows and columns."""
    import torch
    for axis in (0, 1):
        shape = (n, 6) if axis == 0 else (6, n)
        half = [v // 2 + 1 if a == axis else v for a, v in enumerate(shape)]
        x, y = _rand(shape, False, "f64", 1), _rand(tuple(half), True, "f64", 2)
        for fwd, bwd in ((_lib.R2C, _lib.R2C_ADJOINT),):
            ax, _ = _run(fwd, x, half, torch.complex128, [axis], True, 1.0)
            xd = torch.from_numpy(y).cuda()
            gd = torch.zeros(shape, dtype=torch.float64, device="cuda")
            st = [[s * t.element_size() for s in t.stride()] for t in (xd, gd)]
            pl = F.Plan(bwd, list(shape), st[0], st[1], [axis], True)
            pl.execute(xd.data_ptr(), gd.data_ptr(), 1.0, torch.cuda.current_stream().cuda_stream)
            lhs = float(np.sum(ax.real * y.real + ax.imag * y.imag))
            rhs = float(np.sum(x * gd.cpu().numpy()))
            assert abs(lhs - rhs) <= 1e-12 * np.linalg.norm(ax) * np.linalg.norm(y)
        # c2r and its adjoint
        z, _ = _run(_lib.C2R, y, shape, torch.float64, [axis], False, 1.0)
        xd = torch.from_numpy(x).cuda()
        gd = torch.zeros(half, dtype=torch.complex128, device="cuda")
        st = [[s * t.element_size() for s in t.stride()] for t in (xd, gd)]
        pl = F.Plan(_lib.C2R_ADJOINT, list(shape), st[0], st[1], [axis], False)
        pl.execute(xd.data_ptr(), gd.data_ptr(), 1.0, torch.cuda.current_stream().cuda_stream)
        g = gd.cpu().numpy()
        lhs = float(np.sum(z * x))
        rhs = float(np.sum(g.real * y.real + g.imag * y.imag))
        assert abs(lhs - rhs) <= 1e-12 * np.linalg.norm(z) * np.linalg.norm(x)


@pytest.mark.parametrize("n", [10800, 27000, 46305])
def test_four_step(n):
    """Long lengths split into two mixed-radix passes (twiddled column pass, transposing row pass)."""
    x = _rand((3, n), True, "f64", n)
    for fwd in (True, False):
        assert rel_l2(F.c2c(x, [1], fwd, 1.0), oracle.c2c(x, [1], fwd, 1.0)) <= TOL["f64"]
    r = _rand((3, n), False, "f64", n)
    Y = F.r2c(r, [1])
    assert rel_l2(Y, oracle.r2c(r, [1], True, 1.0)) <= TOL["f64"]
    assert rel_l2(F.c2r(Y, n, [1], False, 1.0 / n), r) <= TOL["f64"]


@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("n", [17, 19, 34, 51, 101, 289, 509, 1021, 1999, 2999])
def test_bluestein(n, dt):
    """Chirp-z lengths in one pass: c2c of n, r2c and c2r of 2 n (half length) and n (odd pairs, a last
    row without a partner), rows and columns, and an odd row pitch (no complex words)."""
    import torch
    cdt, rdt = (torch.complex64, torch.float32) if dt == "f32" else (torch.complex128, torch.float64)
    for batch in (1, 6, 7):
        for axis in (0, 1):
            shape = (n, batch) if axis == 0 else (batch, n)
            x = _rand(shape, True, dt, n + batch)
            for fwd in (True, False):
                y, ker = _run(_lib.C2C, x, shape, cdt, [axis], fwd, 0.5)
                assert all(k.startswith("k_fft_mix_blue") for k in ker), (n, axis, ker)
                assert rel_l2(y, oracle.c2c(_wide(x), [axis], fwd, 0.5)) <= TOL[dt], (n, batch, axis, fwd)
            for m in ((n, 2 * n) if n % 2 else (2 * n,)):
                shape = (m, batch) if axis == 0 else (batch, m)
                half = [v // 2 + 1 if a == axis else v for a, v in enumerate(shape)]
                x = _rand(shape, False, dt, m + batch)
                for fwd in (True, False):
                    y, ker = _run(_lib.R2C, x, half, cdt, [axis], fwd, 1.0)
                    assert all(k.startswith("k_fft_mix_blue") for k in ker), (m, axis, ker)
                    assert rel_l2(y, oracle.r2c(_wide(x), [axis], fwd, 1.0)) <= TOL[dt], (m, batch, axis)
                    h = _rand(tuple(half), True, dt, m)
                    z, ker = _run(_lib.C2R, h, shape, rdt, [axis], fwd, 1.0 / m)
                    assert all(k.startswith("k_fft_mix_blue") for k in ker), (m, axis, ker)
                    assert rel_l2(z, oracle.c2r(_wide(h), m, [axis], fwd, 1.0 / m)) <= TOL[dt], (m, batch, axis)
    wide = _rand((5, 2 * n + 3), False, dt, 9)
    for v in (wide[:, :2 * n], wide[:, 1:2 * n + 1], wide[::-1, :n], wide[:, 2 * n::-2][:, :n]):
        assert rel_l2(F.r2c(v, [1], True, 1.0), oracle.r2c(_wide(v), [1], True, 1.0)) <= TOL[dt]
    c = _rand((4, n + 1, 3), True, dt, 10)
    got = F.c2r(c[:, ::-1, :], 2 * n, [1], False, 1.0)
    assert rel_l2(got, oracle.c2r(_wide(c[:, ::-1, :]), 2 * n, [1], False, 1.0)) <= TOL[dt]


@pytest.mark.parametrize("n", [101, 202, 509])
def test_bluestein_adjoint_weights(n):
    test_adjoint_weights(n)
