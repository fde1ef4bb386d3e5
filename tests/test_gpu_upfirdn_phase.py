"""The polyphase kernel with taps in registers (k_upfirdn_phase): sizes with enough whole tiles to take it
(both tile heights), rates below and above one, filters of a few taps and shorter than `up`, the outputs at
both ends, batches.  Reference: the same sums in numpy over every output (FP64, one addition per tap), bar
1e-12 relative L2 as in the upfirdn parity tests; and equality with the sums of a short signal's kernel on
the ends."""
import numpy as np
import pytest

from impulse_amd import _lib, synth
from impulse_amd import signal as S
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    import torch   # before the library: both then share one HIP runtime
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    yield
    torch.cuda.synchronize()


def _sums(t, h, up, down):
    nt, nh = len(t), len(h)
    nout = -(-((nt - 1) * up + nh) // down)
    m = np.arange(nout, dtype=np.int64) * down
    q, r = m // up, m % up
    taps = np.zeros((-(-nh // up) + 1) * up)
    taps[:nh] = h
    y = np.zeros(nout)
    for l in range(-(-nh // up)):
        at = q - l
        ok = (at >= 0) & (at < nt)
        y += np.where(ok, t[np.clip(at, 0, nt - 1)], 0.0) * taps[r + l * up]
    return y


@pytest.mark.parametrize("nt,nh,up,down,batch", [(1_100_003, 81, 4, 1, 1), (3_000_001, 41, 1, 2, 1), (1_600_000, 61, 3, 2, 1),
                                                 (1_400_001, 1601, 160, 147, 1), (900_000, 441, 320, 441, 1),
                                                 (1_000_000, 100, 147, 160, 1), (700_000, 7, 1, 1, 3), (2_100_000, 1, 5, 3, 1),
                                                 (300_000, 900, 512, 511, 2), (500_000, 33, 513, 512, 1)])
def test_all_outputs(nt, nh, up, down, batch):
    import torch
    t = synth.uniform((batch, nt), -1.0, 1.0, seed=nt % 1000)
    h = synth.uniform(nh, -1.0, 1.0, seed=nh)
    y = S.UpfirdnPlan(nt, h, up, down, batch, _lib.UPFIRDN_DIRECT).execute(torch.from_numpy(t).cuda()).cpu().numpy()
    for b in range(batch):
        assert rel_l2(y[b], _sums(t[b], h, up, down)) <= 1e-12
    # the first outputs are those of a short signal that starts alike
    short = S.upfirdn(t[0, :4096], h, up, down, _lib.UPFIRDN_DIRECT)
    same = (4096 - 1) * up // down
    assert np.array_equal(y[0, :same], short[:same])
