"""The fused FFT convolution (conv.hip) at the edges of its kernels: images of one row or column, odd
widths (rows that are not aligned to pairs), kernels of even size, rows of several images in one
workgroup, image chunks of the kernel gradient, the longest columns of the fused path and the first
beyond it.  The reference is the same sums by numpy's FP64 FFT on a grid with no wrap-around; its own
rounding is ~1e-15, and the bar is the 1e-12 of the engine's parity tests (float32 arrays: each output
is the FP64 value rounded once, 2^-24, and the FP64 error)."""
import numpy as np
import pytest

from impulse_amd import synth
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu
TOL = {"f64": 1e-12, "f32": 2.0 ** -24 + 1e-12}


@pytest.fixture(scope="module", autouse=True)
def _device():
    import torch   # before the library: both then share one HIP runtime
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    yield
    torch.cuda.synchronize()


def _reference(x, k, g):
    (B, H, W), (KH, KW) = x.shape, k.shape
    s = (H + KH - 1, W + KW - 1)
    cy, cx = (KH - 1) // 2, (KW - 1) // 2
    kf = np.fft.rfft2(k, s)
    xf = np.fft.rfft2(x, s)
    y = np.fft.irfft2(xf * kf, s)[:, cy:cy + H, cx:cx + W]
    full = np.zeros((B,) + s)
    full[:, cy:cy + H, cx:cx + W] = g
    gf = np.fft.rfft2(full)
    gx = np.fft.irfft2(gf * np.conj(kf), s)[:, :H, :W]
    gk = np.fft.irfft2(np.sum(gf * np.conj(xf), axis=0), s)[:KH, :KW]
    return y, gx, gk


@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("shape", [(1, 1, 1, 1, 1), (5, 1, 17, 1, 4), (3, 19, 1, 6, 1), (9, 3, 5, 2, 2),
                                   (2, 33, 47, 8, 9), (17, 40, 61, 7, 12), (3, 200, 77, 31, 30), (1, 479, 300, 5, 63),
                                   (2, 64, 2561, 3, 3), (1, 2529, 40, 63, 5), (1, 2555, 24, 12, 5)])
def test_shapes(shape, dt):
    import torch
    from impulse_amd import autograd as AG
    B, H, W, KH, KW = shape
    npdt = np.float32 if dt == "f32" else np.float64
    x = synth.uniform((B, H, W), 0.0, 1.0, seed=1).astype(npdt)
    k = synth.normal((KH, KW), seed=2).astype(npdt)
    g = synth.normal((B, H, W), seed=3).astype(npdt)
    xd, kd = torch.from_numpy(x).cuda().requires_grad_(), torch.from_numpy(k).cuda().requires_grad_()
    y = AG.fft_conv2d(xd, kd)
    gx, gk = torch.autograd.grad(y, (xd, kd), torch.from_numpy(g).cuda())
    ry, rgx, rgk = _reference(x.astype(np.float64), k.astype(np.float64), g.astype(np.float64))
    for name, a, b in (("y", y.detach(), ry), ("gx", gx, rgx), ("gk", gk, rgk)):
        assert rel_l2(a.cpu().numpy(), b) <= TOL[dt], (name, shape)


def test_single_gradients_and_separate_images():
    """Each gradient alone equals the pair, and an image with NaN leaves the others' outputs as they were."""
    import torch
    from impulse_amd import autograd as AG
    x = torch.from_numpy(synth.uniform((4, 30, 41), 0.0, 1.0, seed=4)).cuda()
    k = torch.from_numpy(synth.normal((5, 6), seed=5)).cuda()
    g = torch.from_numpy(synth.normal((4, 30, 41), seed=6)).cuda()
    xa, ka = x.clone().requires_grad_(), k.clone().requires_grad_()
    gx, gk = torch.autograd.grad(AG.fft_conv2d(xa, ka), (xa, ka), g)
    assert torch.equal(torch.autograd.grad(AG.fft_conv2d(xa, k), xa, g)[0], gx)
    assert torch.equal(torch.autograd.grad(AG.fft_conv2d(x, ka), ka, g)[0], gk)
    y = AG.fft_conv2d(x, k)
    bad = x.clone()
    bad[2, 3, 4] = float("nan")
    z = AG.fft_conv2d(bad, k)
    keep = [0, 1, 3]
    assert torch.equal(z[keep], y[keep]) and bool(torch.isnan(z[2]).any())
