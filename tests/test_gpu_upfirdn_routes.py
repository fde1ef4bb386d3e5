"""Upfirdn on both sides of the rule for the polyphase kernel with taps in registers: every output against
the same sums in numpy (FP64, one addition per tap) at 1e-12 relative L2, the bar of the upfirdn parity
tests, on the first and the last signal of a batch.  tests/test_upfirdn_host.py checks which kernel each
of these sizes takes."""
import numpy as np
import pytest

from impulse_amd import _lib, synth
from impulse_amd import signal as S
from tests.conftest import rel_l2
from tests.upfirdn_phase_cases import PHASE, TILE

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


@pytest.mark.parametrize("nt,nh,up,down,batch", [c[:5] for c in PHASE] + TILE)
def test_all_outputs(nt, nh, up, down, batch):
    import torch
    t = synth.uniform((batch, nt), -1.0, 1.0, seed=nt % 1000)
    h = synth.uniform(nh, -1.0, 1.0, seed=nh)
    y = S.UpfirdnPlan(nt, h, up, down, batch, _lib.UPFIRDN_DIRECT).execute(torch.from_numpy(t).cuda()).cpu().numpy()
    for b in sorted({0, batch // 2, batch - 1}):
        assert rel_l2(y[b], _sums(t[b], h, up, down)) <= 1e-12, b
