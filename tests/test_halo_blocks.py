"""The halo gridder's persistent workgroups of one wavefront: whole fours a CU
where more than four fit, so that its SIMDs hold the same number (over a
stand-in for the HIP runtime, 256 CUs; no GPU)."""
import pytest

import hipstub


@pytest.mark.parametrize("fit,run", [(1, 1), (3, 3), (4, 4), (5, 4), (7, 4), (8, 8), (13, 12)])
def test_whole_fours(tmp_path, fit, run):
    out = hipstub.run(tmp_path, f"""
stub.stub_per_cu({fit})
buf = C.create_string_buffer(64 * 64 * 8)
at = C.addressof(buf)
geom = _lib.Geom(at, at, 4, 5, 1.0, 1.0, 64, 64)
gcf = _lib.Gcf(at, at, at, 64, 0, at, 0, 1, 64)
plan = C.c_void_p()
assert h.rcg_tiled_plan_create_ex(C.byref(geom), 1, 32, 512, 32, 1, C.byref(plan)) == 0
assert h.rcg_grid_tiled_f32(plan, C.byref(gcf), at, at, None) == 0
print(stub.stub_last_grid(64) // 256)
""")
    assert int(out) == run
