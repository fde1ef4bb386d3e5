"""Every radix that the mixed-radix pass kernel is given in each place -- 2, 3, 5, 6, 7 and 9 to 15 first
(the factoring never starts with 4, 8 or 16), 2 to 16 between and last -- and two to six stages: complex
transforms of these lengths, even real ones of twice and odd real ones of the odd lengths, rows and columns,
both directions, against the long-double oracle at 1e-12, the bar of the parity tests.
tests/test_mix_lengths_host.py checks that the lengths cover what the factoring gives."""
import numpy as np
import pytest

import oracle
from impulse_amd import synth
from impulse_amd import fft as F
from tests.conftest import rel_l2
from tests.mix_lengths import LENGTHS

pytestmark = pytest.mark.gpu
TOL = 1e-12


@pytest.fixture(scope="module", autouse=True)
def _device():
    import torch   # before the library: both then share one HIP runtime
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    yield
    torch.cuda.synchronize()


@pytest.mark.parametrize("n", LENGTHS)
def test_complex(n):
    z = synth.complex_normal((3, n), seed=n)
    zt = np.ascontiguousarray(z.T)
    for forward in (True, False):
        want = oracle.c2c(z, [1], forward)
        assert rel_l2(F.c2c(z, [1], forward), want) <= TOL
        assert rel_l2(F.c2c(zt, [0], forward).T, want) <= TOL


@pytest.mark.parametrize("n", [2 * n for n in LENGTHS] + [n for n in LENGTHS if n % 2])
def test_real(n):
    x = synth.uniform((3, n), -1.0, 1.0, seed=n)
    want = oracle.r2c(x, [1])
    assert rel_l2(F.r2c(x, [1]), want) <= TOL
    assert rel_l2(F.r2c(np.ascontiguousarray(x.T), [0]).T, want) <= TOL
    assert rel_l2(F.c2r(want, n, [1], False, 1.0 / n), x) <= TOL
    assert rel_l2(F.c2r(np.ascontiguousarray(want.T), n, [0], False, 1.0 / n).T, x) <= TOL
