"""Launch shapes of the convolution's kernel gradient (no GPU): the stand-in HIP runtime of
tests/cpp/hip_stand_in.cpp."""
import pytest


@pytest.mark.parametrize("batch,size,k,threads", [(64, 16, 3, 48), (100, 28, 7, 64), (2000, 16, 3, 48), (8000, 16, 3, 48),
                                                  (4000, 8, 3, 24), (256, 64, 9, 64)])
def test_small_images_in_many_chunks(hip_host, batch, size, k, threads):
    """A workgroup sums its chunk's images one after the other: batches of small images take more chunks
    the more images they hold, and short columns take a thread per butterfly up to a wavefront."""
    cols = hip_host(f"""
h = ctypes.c_void_p()
rc = L.impulse_fft_conv2d_create(ctypes.byref(h), {batch}, {size}, {size}, {k}, {k}, 1)
assert rc == 0, L.impulse_fft_last_error()
launches()
assert L.impulse_fft_conv2d_backward(h, 1 << 30, 1 << 31, 1 << 32, 0, 1 << 33, None) == 0
report([l for l in launches() if "k_conv_cols" in l[0]])
""")
    gk = [l for l in cols if "k_conv_colsILi2E" in l[0]]
    final = [l for l in cols if "k_conv_colsILi3E" in l[0]]
    assert len(gk) == 1 and len(final) == 1
    groups = int(final[0][1])                      # column blocks
    per_block = int(gk[0][1]) // groups            # workgroups per block: parts times chunks
    assert int(gk[0][3]) >= threads
    assert per_block * (batch ** 0.5) >= batch     # at most about sqrt(batch) images each
