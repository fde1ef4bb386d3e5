"""Which direct kernel an upfirdn plan launches (no GPU): the stand-in HIP runtime of
tests/cpp/hip_stand_in.cpp."""
import pytest

from tests.upfirdn_phase_cases import PHASE, TILE


def _launch(hip_host, nt, nh, up, down, batch):
    got = hip_host(f"""
import array
taps = array.array("d", [1.0] * {nh})
h = ctypes.c_void_p()
rc = L.impulse_fft_upfirdn_create(ctypes.byref(h), {batch}, {nt}, taps.buffer_info()[0], {nh}, {up}, {down}, 1)
assert rc == 0, L.impulse_fft_last_error()
launches()
assert L.impulse_fft_upfirdn_execute(h, 1 << 40, 1 << 41, None) == 0
report(launches())
""")
    assert len(got) == 1
    return got[0]


@pytest.mark.parametrize("nt,nh,up,down,batch,outputs", PHASE)
def test_long_signals_take_the_phase_kernel(hip_host, nt, nh, up, down, batch, outputs):
    assert f"k_upfirdn_phaseILi{outputs}E" in _launch(hip_host, nt, nh, up, down, batch)[0]


@pytest.mark.parametrize("nt,nh,up,down,batch", TILE)
def test_short_signals_keep_the_tile_kernel(hip_host, nt, nh, up, down, batch):
    """Batches of signals whose ends are more than a 64th of their outputs, few whole tiles, and rates over
    512."""
    name = _launch(hip_host, nt, nh, up, down, batch)[0]
    assert "k_upfirdn_tile" in name or "k_upfirdn_direct" in name
