"""Non-smooth lengths from 3,841 to 4,096, whose padded transform of up to 8,192 points is the longest of the
one-pass mixed-radix Bluestein kernel: complex and real, rows and columns, both directions, float arrays,
against the oracle at 1e-12 (float arrays: 1e-6), the bars of the parity tests."""
import numpy as np
import pytest

import oracle
from impulse_amd import synth
from impulse_amd import fft as F
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    import torch   # before the library: both then share one HIP runtime
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    yield
    torch.cuda.synchronize()


@pytest.mark.parametrize("n", [3841, 3851, 3889, 3899, 4093])
@pytest.mark.parametrize("batch", [1, 3])
def test_lengths(n, batch):
    re, im = (synth.uniform((batch, n), -1.0, 1.0, seed=n + k) for k in (0, 1))
    z = re + 1j * im
    for forward in (True, False):
        assert rel_l2(F.c2c(z, [1], forward), oracle.c2c(z, [1], forward)) <= 1e-12
        zt = np.ascontiguousarray(z.T)
        assert rel_l2(F.c2c(zt, [0], forward), oracle.c2c(zt, [0], forward)) <= 1e-12
        assert rel_l2(F.c2c(z.astype(np.complex64), [1], forward), oracle.c2c(z.astype(np.complex64).astype(z.dtype), [1], forward)) <= 1e-6
    for m in (n, 2 * n):   # odd rows in pairs; even rows at half length
        x = synth.uniform((batch, m), -1.0, 1.0, seed=m)
        y = F.r2c(x, [1])
        want = oracle.r2c(x, [1])
        assert rel_l2(y, want) <= 1e-12
        assert rel_l2(F.c2r(want, m, [1], False, 1.0 / m), x) <= 1e-12
