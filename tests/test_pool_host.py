"""The device memory kept between MS4 calls, over a stand-in for the HIP
runtime (no GPU): it is given back to any allocation of the library that
would fail without it, and no failure leaves a HIP error behind."""
import pytest

import hipstub

# a call whose points all lie outside the grid (no kernel runs here, so none
# is found inside): its buffers stay with the pool
KEEP = """
import numpy as np
from rc_amd import ms4, synth
vc, gcf, _ = synth.random_small(1, grid_size=64, chunks=2000, ts_ch=20)
ms4.grid(vc, gcf, 64)
kept = stub.stub_live()
assert kept > 1 << 20
plan = C.c_void_p()
def make_plan():
    geom = _lib.Geom(0x1000, 0x1000, 4000, 50, 1.0, 1.0, 256, 256)
    return h.rcg_tiled_plan_create_ex(C.byref(geom), 1, 32, 512, 16, 0, C.byref(plan))
"""


def test_plan_gets_what_the_pool_keeps(tmp_path):
    out = hipstub.run(tmp_path, KEEP + """
assert make_plan() == 0
need = stub.stub_live() - kept
h.rcg_tiled_plan_destroy(plan)
assert stub.stub_live() == kept
stub.stub_limit(kept + need - 1)       # one byte short beside the kept memory
assert make_plan() == 0 and stub.stub_live() == need
assert stub.hipGetLastError() == 0
h.rcg_tiled_plan_destroy(plan)
ms4.grid(vc, gcf, 64)                  # and the calls go on
assert stub.stub_live() == kept
print("ok")
""")
    assert out.split() == ["ok"]


@pytest.mark.parametrize("size,fits", [(600, True), (1 << 20, False)])
def test_deconvolve_gets_what_the_pool_keeps(tmp_path, size, fits):
    """Three images and the scratch: 600^2 fits without the kept memory;
    2^20 squared (8 TiB) does not, and is refused before the images are
    touched."""
    out = hipstub.run(tmp_path, KEEP + f"""
size = {size}
need = 3 * 8 * size * size + h.rcg_hogbom_scratch_bytes()
stub.stub_limit(need + kept // 2 if {fits} else kept + (1 << 20))
n = size * size if {fits} else 1
a = [np.zeros(n) for _ in range(3)]
h.deconvolve(a[0].ctypes.data, a[1].ctypes.data, a[2].ctypes.data, size, size, 5, 0.1, 0.0)
assert h.rcg_last_error() == (0 if {fits} else 3)
assert stub.hipGetLastError() == 0
assert stub.stub_live() == 0           # nothing kept, nothing lost
print("ok")
""")
    assert out.split() == ["ok"]


def test_calls_without_host_memory(tmp_path):
    """Every C++ allocation of a call in turn fails: the call ends with an
    error or does without, nothing is lost, and the next call works.  (An
    exception that left a C entry point, a destructor or a thread would end
    the process.)"""
    out = hipstub.run(tmp_path, KEEP + """
h.rcg_shutdown()
assert stub.stub_live() == 0
failed = 0
for n in range(1, 400):
    stub.stub_fail_new(n)
    try:
        ms4.grid(vc, gcf, 64)
    except _lib.RcgError:
        assert h.rcg_last_error() in (2, 3)
        failed += 1
    left = stub.stub_new_left()        # 0: the n-th allocation was reached
    stub.stub_fail_new(0)
    ms4.grid(vc, gcf, 64)
    assert stub.stub_live() == kept
    if n % 2:
        h.rcg_shutdown()
        assert stub.stub_live() == 0
    if left:
        break
assert 1 <= failed < n < 399, (failed, n)
print("ok")
""")
    assert out.split() == ["ok"]
