"""DCT and DST of arrays over 2 GiB in one kernel per axis (k_r2r_mix with offsets from a workgroup's own
first line): contiguous rows, padded rows whose workgroups pass from one slab into the next, rows in
reverse order, and lines across memory, in place and out of place.  Every line goes through the same
arithmetic as in a small array, which other tests compare with the oracle, so lines from the start, the
2 GiB mark, the slab ends and the end of the large array equal their small transform bit for bit."""
import ctypes

import pytest

from impulse_amd import _lib
from impulse_amd._lib import check, lib, sizes, strides as bstrides

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    import torch   # before the library: both then share one HIP runtime
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    yield
    torch.cuda.synchronize()
    torch.cuda.empty_cache()


def _run(kind, t, shape, st, axis, src, dst, launches=None):
    """src, dst: addresses of element 0; strides in elements"""
    import torch
    L = lib()
    h = ctypes.c_void_p()
    b = bstrides([8 * s for s in st])
    check(L.impulse_fft_r2r_plan_create(ctypes.byref(h), kind, t, 1, _lib.F64, len(shape), sizes(shape), b, b, 1,
                                        sizes([axis])))
    if launches is not None:
        assert L.impulse_fft_plan_num_launches(h) == launches
    check(L.impulse_fft_execute(h, src, dst, 0.5, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    check(L.impulse_fft_plan_destroy(h))


def _small(kind, t, x, axis):
    import torch
    x = x.contiguous()
    y = torch.empty_like(x)
    st = [int(s) for s in x.stride()]
    _run(kind, t, list(x.shape), st, axis, x.data_ptr(), y.data_ptr())
    return y


def _data(n, seed):
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.rand(n, generator=g, device="cuda", dtype=torch.float64) - 0.5


@pytest.mark.parametrize("kind,t", [(_lib.DCT, 2), (_lib.DST, 3), (_lib.DCT, 4)])
def test_rows(kind, t):
    import torch
    rows, n = 33000, 8192
    x = _data(rows * n, t).view(rows, n)
    y = torch.zeros_like(x)
    _run(kind, t, [rows, n], [n, 1], 1, x.data_ptr(), y.data_ptr(), 1)
    pick = torch.tensor([0, 1, 32766, 32767, 32768, rows - 2, rows - 1], device="cuda")
    want = _small(kind, t, x[pick], 1)
    assert torch.equal(y[pick], want)
    # the same rows last to first: element 0 is the last row's
    y.zero_()
    last = (rows - 1) * n * 8
    _run(kind, t, [rows, n], [-n, 1], 1, x.data_ptr() + last, y.data_ptr() + last, 1)
    assert torch.equal(y[pick], want)
    assert bool((y.abs().amax(1) > 0).all())


@pytest.mark.parametrize("kind,t", [(_lib.DST, 2), (_lib.DCT, 3), (_lib.DST, 4)])
def test_padded_short_rows_in_place(kind, t):
    import torch
    a, b, n, pad = 3, 1500001, 64, 65
    x = _data(a * b * pad, t).view(a, b, pad)
    before = x.clone()
    pick = torch.tensor([0, 1, 62, 63, 64, b // 2, b - 65, b - 64, b - 2, b - 1], device="cuda")
    _run(kind, t, [a, b, n], [b * pad, pad, 1], 2, x.data_ptr(), x.data_ptr(), 1)
    for s in range(a):
        assert torch.equal(x[s, pick, :n], _small(kind, t, before[s, pick, :n], 1)), s
    assert torch.equal(x[:, :, n:], before[:, :, n:])
    assert bool((x[:, :, :n] != before[:, :, :n]).any(-1).all())


@pytest.mark.parametrize("kind,t", [(_lib.DCT, 2), (_lib.DST, 3), (_lib.DST, 4)])
def test_columns(kind, t):
    import torch
    a, n, c = 5, 1024, 60000
    x = _data(a * n * c, t).view(a, n, c)
    y = torch.zeros_like(x)
    _run(kind, t, [a, n, c], [n * c, c, 1], 1, x.data_ptr(), y.data_ptr(), 1)
    pick = torch.tensor([0, 1, 7, 8, c // 2, c - 2, c - 1], device="cuda")
    for s in range(a):
        assert torch.equal(y[s][:, pick], _small(kind, t, x[s][:, pick], 0)), s
    assert bool((y.abs().amax(1) > 0).all())
