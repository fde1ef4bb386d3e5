"""Host side of ragged batches (no GPU): what creating one allocates, and what a failed allocation
leaves behind.  The HIP runtime is the stand-in of tests/cpp/hip_stand_in.cpp."""
import pytest

CREATE = """
def create(lengths, ins, outs):
    h = ctypes.c_void_p()
    return L.impulse_fft_ragged_create(ctypes.byref(h), len(lengths), _lib.sizes(lengths), _lib.sizes(ins),
                                       _lib.sizes(outs), 1), h
"""


@pytest.mark.parametrize("gap", [8 << 30, 1 << 40])
def test_sparse_offsets(hip_host, gap):
    # Two short signals far apart in their buffers: the host memory of a batch follows the samples
    # it holds, not the distance between them.
    kib = hip_host(CREATE + f"""
import resource
rc, h = create([1000, 4099], [0, {gap}], [0, {gap}])
assert rc == 0, L.impulse_fft_last_error()
assert L.impulse_fft_ragged_configure(h, 512, 4096, 0, 0) == 0
report(resource.getrusage(resource.RUSAGE_SELF).ru_maxrss)
""")
    assert kib < 256 << 10
