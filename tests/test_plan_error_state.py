"""A plan that cannot be made leaves no HIP error behind: the next launch of
a caller that goes on without it (the FP64 Imager and the MS4 and MS6 calls
take the plain gridder) would report the old one."""
import pytest

import hipstub


@pytest.mark.parametrize("tile,max_support,layout", [(16, 8, 0), (32, 16, 0), (64, 40, 0),
                                                     (32, 100, 0), (16, 16, 1), (32, 32, 1)])
def test_failed_plan_leaves_no_hip_error(tmp_path, tile, max_support, layout):
    out = hipstub.run(tmp_path, f"""
geom = _lib.Geom(0x1000, 0x1000, 4000, 50, 1.0, 1.0, 256, 256)
plan = C.c_void_p()
make = lambda: h.rcg_tiled_plan_create_ex(C.byref(geom), 1, {tile}, 512, {max_support}, {layout},
                                          C.byref(plan))
assert make() == 0 and plan.value
whole = stub.stub_live()
assert h.rcg_tiled_plan_destroy(plan) == 0 and stub.stub_live() == 0
for part in range(8):  # every allocation in turn is the one that fails
    stub.stub_limit(whole * part // 8)
    assert make() == 3 and not plan.value  # RCG_ERR_NOMEM
    assert stub.stub_live() == 0
    assert stub.hipGetLastError() == 0, part
print("ok")
""")
    assert out.split() == ["ok"]
