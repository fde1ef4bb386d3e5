"""DCT and DST of types 2-4 at even lengths in one kernel per axis (k_r2r_mix): the smallest lengths
(N/2 = 1, one radix), powers of two (padded LDS rows), composite and prime radices, the longest length of
the path and the first beyond it; lines along the unit-stride axis with aligned and unaligned pairs,
lines across memory with few and many neighbours, reversed and strided views, `ortho`, in place.  Against
the oracle's long-double sums at 1e-12, the parity bar of the DCT tests (long lengths against the
oracle's FFT-based pair: the inverse type gives 2 N x back)."""
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


def _launches(sine, t, shape, axes):
    from impulse_amd import _lib
    st, acc = [0] * len(shape), 8
    for d in range(len(shape) - 1, -1, -1):
        st[d] = acc
        acc *= shape[d]
    p = F.Plan(_lib.DST if sine else _lib.DCT, list(shape), st, st, list(axes), True, r2r_type=t)
    return p.num_launches


@pytest.mark.parametrize("t", [2, 3, 4])
@pytest.mark.parametrize("sine", [False, True])
def test_lengths_rows_and_columns(t, sine):
    ref, run = (oracle.dst, F.dst) if sine else (oracle.dct, F.dct)
    for n, batches in ((2, (1, 3, 130)), (4, (3,)), (6, (130,)), (10, (3,)), (14, (1,)), (22, (3,)), (26, (7,)), (32, (130,)),
                       (34, (3,)), (64, (3,)), (66, (70,)), (120, (3,)), (242, (1,)), (250, (3,)), (256, (3,)), (338, (1,))):
        for batch in batches:
            x = synth.uniform((batch, n), -1.0, 1.0, seed=n + batch)
            for ortho in (False, True):
                assert rel_l2(run(x, [1], t, 0.5, ortho), ref(x, [1], t, 0.5, ortho)) <= TOL, (n, batch, ortho, "rows")
                xc = np.ascontiguousarray(x.T)
                assert rel_l2(run(xc, [0], t, 0.5, ortho), ref(xc, [0], t, 0.5, ortho)) <= TOL, (n, batch, ortho, "cols")
    assert _launches(sine, t, (3, 1000), [0, 1][1:]) == 1 and _launches(sine, t, (1000, 3), [0]) == 1


@pytest.mark.parametrize("t", [2, 3, 4])
@pytest.mark.parametrize("sine", [False, True])
def test_views(t, sine):
    ref, run = (oracle.dst, F.dst) if sine else (oracle.dct, F.dct)
    a = synth.uniform((5, 61, 40), -1.0, 1.0, seed=7)
    for v, ax in ((a[:, ::2, :][:, :30, :], [1]), (a[::-1, 59::-1, 1:8], [1]), (a[:, 1:, 1:39], [2]), (a[:, :, ::-2], [2]),
                  (a[:, :60, :38], [2, 1]), (a.transpose(2, 0, 1)[:, :, :60], [0, 2])):
        assert rel_l2(run(v, ax, t, 1.0, True), ref(np.ascontiguousarray(v), ax, t, 1.0, True)) <= TOL, (v.strides, ax)
    b = a[:, :60, :].copy()
    want = ref(b, [1, 2], t, 0.25, False)
    run(b, [1, 2], t, 0.25, False, out=b)
    assert rel_l2(b, want) <= TOL


@pytest.mark.parametrize("n", [6250, 8190, 8192, 8194, 8400])
def test_long(n):
    """N/2 = 3125 (five stages), 4095, 4096 (the longest in one kernel), and two beyond it."""
    for axis in (0, 1):
        x = synth.uniform((n, 5) if axis == 0 else (5, n), -1.0, 1.0, seed=n)
        for sine in (False, True):
            run = F.dst if sine else F.dct
            for t, u in ((2, 3), (4, 4)):
                y = run(x, [axis], t)
                assert rel_l2(run(y, [axis], u, 0.5 / n), x) <= TOL, (n, axis, sine, t)
                # one coefficient against its sum
                k, j = 17, np.arange(n)
                ph = (2 * j + 1) * ((k + 1 if sine else k) if t == 2 else 2 * k + 1) % (4 * n if t == 2 else 8 * n)
                w = (np.sin if sine else np.cos)(ph * (np.pi / ((2 if t == 2 else 4) * n)))
                got = y[k] if axis == 0 else y[:, k]
                want = 2.0 * (np.tensordot(w, x, (0, 0)) if axis == 0 else x @ w)
                assert np.max(np.abs(got - want)) <= 1e-10 * np.sqrt(n), (n, axis, sine, t)
