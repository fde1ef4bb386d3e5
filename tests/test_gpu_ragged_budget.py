"""The LDS budget a ragged batch starts with follows from its lengths: the small one where every length
splits into its tiles (up to 2048 x 1024 complex points), a larger one where one does not, and the bins
are the FP64 transform's either way (1e-12, the bar of the ragged parity tests; the reference is numpy's
FP64 rfft, itself within 1e-15)."""
import numpy as np
import pytest

from impulse_amd import synth
from impulse_amd.ragged import RaggedBatch
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    import torch   # before the library: both then share one HIP runtime
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    yield
    torch.cuda.synchronize()


# 2^22: M = 2^21 = 2048 x 1024, the longest power of two of the small budget; 2^23 is beyond it
@pytest.mark.parametrize("longest,points", [(2048, 2048), (1 << 22, 2048), (1 << 23, 4096)])
def test_starting_budget(longest, points):
    import torch
    lengths = [97, 1000, longest]
    b = RaggedBatch(lengths)
    assert b.info()["lds_points"] == points
    x = synth.uniform(b.in_elems, -1.0, 1.0, seed=longest % 97).astype(np.float32)
    y = b.execute(torch.from_numpy(x).cuda(), torch.empty(b.out_elems, dtype=torch.complex128, device="cuda"))
    torch.cuda.synchronize()
    for n, i, v in zip(lengths, b.in_offsets, b.output_views(y)):
        assert rel_l2(v.cpu().numpy(), np.fft.rfft(x[i:i + n].astype(np.float64))) <= 1e-12, n


@pytest.mark.parametrize("fill,points", [(0, 8192), (767, 8192), (768, 2048)])
def test_single_phase_budget(fill, points):
    """A Bluestein length over the small budget's points (2206 = 2 * 1103) in a batch of at most three signals a
    CU starts with the largest budget; one signal more, and it does not."""
    import torch
    lengths = [96] * fill + [2206]
    b = RaggedBatch(lengths)
    assert b.info()["lds_points"] == points
    x = synth.uniform(b.in_elems, -1.0, 1.0, seed=fill).astype(np.float32)
    y = b.execute(torch.from_numpy(x).cuda(), torch.empty(b.out_elems, dtype=torch.complex128, device="cuda"))
    torch.cuda.synchronize()
    for n, i, v in list(zip(lengths, b.in_offsets, b.output_views(y)))[-3:]:
        assert rel_l2(v.cpu().numpy(), np.fft.rfft(x[i:i + n].astype(np.float64))) <= 1e-12, n
