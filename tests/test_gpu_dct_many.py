"""DCT and DST of many short lines and of few long ones, where a line takes more threads than its
butterflies need (k_r2r_mix): from two to 512 threads a line, rows and columns, against the oracle's
long-double sums on lines at workgroup ends, at 1e-12, the parity bar of the DCT tests."""
import numpy as np
import pytest

import oracle
from impulse_amd import synth
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


@pytest.mark.parametrize("n", [10, 14, 16, 18, 26, 30, 32, 50, 64, 90])
@pytest.mark.parametrize("lines", [37, 1000, 20011])
def test_short_lines(n, lines):
    pick = sorted({0, 1, 2, 15, 16, 31, 32, 33, lines // 2, lines - 2, lines - 1})
    x = synth.uniform((lines, n), -1.0, 1.0, seed=n + lines)
    xc = np.ascontiguousarray(x.T)
    for sine in (False, True):
        ref, run = (oracle.dst, F.dst) if sine else (oracle.dct, F.dct)
        for t in (2, 3, 4):
            want = ref(np.ascontiguousarray(x[pick]), [1], t, 0.5, True)
            assert rel_l2(run(x, [1], t, 0.5, True)[pick], want) <= TOL, (sine, t, "rows")
            assert rel_l2(run(xc, [0], t, 0.5, True).T[pick], want) <= TOL, (sine, t, "cols")


@pytest.mark.parametrize("n", [1000, 2048, 2430, 6250])
@pytest.mark.parametrize("lines", [1, 3, 130])
def test_few_long_lines(n, lines):
    x = synth.uniform((lines, n), -1.0, 1.0, seed=n + lines)
    for sine in (False, True):
        ref, run = (oracle.dst, F.dst) if sine else (oracle.dct, F.dct)
        for t in (2, 3, 4):
            want = ref(np.ascontiguousarray(x[-1:]), [1], t, 1.0, False)
            assert rel_l2(run(x, [1], t, 1.0, False)[-1:], want) <= TOL, (sine, t, "rows")
            got = run(np.ascontiguousarray(x.T), [0], t, 1.0, False).T[-1:]
            assert rel_l2(got, want) <= TOL, (sine, t, "cols")
