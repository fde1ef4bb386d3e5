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
def peak():   # address space of this process, KiB
    return next(int(l.split()[1]) for l in open("/proc/self/status") if l.startswith("VmPeak"))
rc, h = create([1000, 4099], [0, 8192], [0, 8192])   # the same batch close together
before = peak()
rc, h = create([1000, 4099], [0, {gap}], [0, {gap}])
assert rc == 0, L.impulse_fft_last_error()
assert L.impulse_fft_ragged_configure(h, 512, 4096, 0, 0) == 0
report(peak() - before)
""")
    assert kib < 64 << 10


def test_budget_follows_device_memory(hip_host):
    # The starting budget keeps a workspace for the transforms of 8,192 points, the largest one holds
    # them in LDS: where the workspace does not fit, the batch is created without it.
    roomy, tight = hip_host(CREATE + """
n = [16384] * 1000 + [4096] * 4000
ins, outs = [16384 * i for i in range(5000)], [8193 * i for i in range(5000)]
got = []
for limit in (1 << 40, 64 << 20):
    S.standin_limit(limit)
    rc, h = create(n, ins, outs)
    assert rc == 0, L.impulse_fft_last_error()
    t, b, w = ctypes.c_int(), ctypes.c_int(), ctypes.c_size_t()
    L.impulse_fft_ragged_info(h, ctypes.byref(t), ctypes.byref(b), None, None, None, None, ctypes.byref(w))
    got.append([t.value, b.value, w.value, S.standin_used()])
    L.impulse_fft_ragged_destroy(h)
report(got)
""")
    assert roomy[1] == 2048 and roomy[2] >= 1000 * 8192 * 16
    assert tight[1] == 8192 and tight[2] < 1024


def test_refused_configuration(hip_host):
    # A configuration whose workspace does not fit is refused, and so are executes from then on until
    # one that fits is set; nothing is launched on buffers that are gone.
    got = hip_host(CREATE + """
n = [16384] * 1000
ins, outs = [16384 * i for i in range(1000)], [8193 * i for i in range(1000)]
S.standin_limit(64 << 20)
rc, h = create(n, ins, outs)
assert rc == 0
x, y = 1 << 40, 1 << 41
run = lambda: L.impulse_fft_ragged_execute(h, x, y, 1.0, None)
got = [run()]
launches()
got.append(L.impulse_fft_ragged_configure(h, 256, 2048, 0, 3))
got.append(run())
got.append(len(launches()))
got.append(L.impulse_fft_ragged_configure(h, 1024, 8192, 0, 0))
got.append(run())
report(got)
""")
    NOMEM = 2
    assert got[0] == 0 and got[1] == NOMEM
    assert got[2] != 0 and got[3] == 0
    assert got[4] == 0 and got[5] == 0


def test_tuning_passes_over_what_does_not_fit(hip_host):
    # The candidates whose workspace does not fit are left out, as those with no split are.
    rc, budget, run = hip_host(CREATE + """
n = [16384] * 1000
ins, outs = [16384 * i for i in range(1000)], [8193 * i for i in range(1000)]
S.standin_limit(64 << 20)
rc, h = create(n, ins, outs)
assert rc == 0
ms, b = ctypes.c_double(), ctypes.c_int()
rc = L.impulse_fft_ragged_tune(h, 1 << 40, 1 << 41, None, 1, ctypes.byref(ms))
L.impulse_fft_ragged_info(h, None, ctypes.byref(b), None, None, None, None, None)
report([rc, b.value, L.impulse_fft_ragged_execute(h, 1 << 40, 1 << 41, 1.0, None)])
""")
    assert (rc, budget, run) == (0, 8192, 0)


@pytest.mark.parametrize("lengths,points", [
    ("[2048] * 1000", 2048), ("[4096] * 10000", 2048),                       # held by the smallest budget
    ("[8192] * 1", 4096), ("[8192] * 1000", 4096), ("[4095] * 2000", 4096), ("[2047] * 2000", 4096),
    ("[16384] * 30", 2048), ("[16384] * 64", 8192), ("[16384] * 1000", 8192), ("[4100] * 2000", 8192),
    ("[16384] * 1000 + [16386] * 10", 2048),                                 # 8,193 = 3 * 2731: Bluestein beyond 8,192 points
    ("[16384] * 100 + [4096] * 2000", 2048),                                 # mostly short ones
    ("[97] * 5 + [8198]", 2048), ("[97] * 5 + [2206]", 8192), ("[96] * 768 + [2206]", 2048),
])
def test_starting_budget(hip_host, lengths, points):
    """The larger budgets where they hold all of a batch in LDS and are faster on it (256 CUs)."""
    got = hip_host(CREATE + f"""
n = {lengths}
ins, outs = [0] * len(n), [16384 * i for i in range(len(n))]
rc, h = create(n, ins, outs)
assert rc == 0, L.impulse_fft_last_error()
b = ctypes.c_int()
L.impulse_fft_ragged_info(h, None, ctypes.byref(b), None, None, None, None, None)
report(b.value)
""")
    assert got == points


def test_starting_budget_follows_precision(hip_host):
    """A batch starts with the budget of its precision until a configuration is set."""
    got = hip_host(CREATE + """
n = [16384] * 1000
rc, h = create(n, [0] * 1000, [8193 * i for i in range(1000)])
assert rc == 0
def budget():
    b = ctypes.c_int()
    L.impulse_fft_ragged_info(h, None, ctypes.byref(b), None, None, None, None, None)
    return b.value
got = [budget()]
for precision in (1, 0, 1):
    assert L.impulse_fft_ragged_set_precision(h, precision) == 0
    got.append(budget())
assert L.impulse_fft_ragged_configure(h, 512, 4096, 0, 4) == 0
for precision in (0, 1):
    assert L.impulse_fft_ragged_set_precision(h, precision) == 0
    got.append(budget())
report(got)
""")
    assert got == [8192, 2048, 8192, 2048, 4096, 4096]
