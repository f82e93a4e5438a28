"""Which plans degrid by whole windows: those whose items hold points enough
(chunk over the tiles that a window meets) and whose region fits (over a
stand-in for the HIP runtime, no GPU: whole windows are one launch behind the
clearing one, pairs are two)."""
import pytest

import hipstub


@pytest.mark.parametrize("tile,support,chunk,windows", [
    (32, 8, 44, False), (32, 8, 45, True),          # 30 points of 1.48 tiles
    (32, 31, 112, False), (32, 31, 113, True),      # 3.75
    (32, 63, 258, False), (32, 63, 259, True),      # 8.63
    (32, 64, 512, True), (32, 65, 1 << 20, False),  # the region's LDS
    (16, 48, 465, False), (16, 48, 466, True), (16, 63, 512, False), (16, 63, 1024, True),
    (64, 31, 64, False), (64, 31, 65, True), (32, 1, 29, False), (32, 1, 30, True)])
def test_rule(tmp_path, tile, support, chunk, windows):
    out = hipstub.run(tmp_path, f"""
buf = C.create_string_buffer(64 * 64 * 8)
at = C.addressof(buf)
geom = _lib.Geom(at, at, 4, 5, 1.0, 1.0, 64, 64)
gcf = _lib.Gcf(at, at, at, 64, 0, at, 0, 1, 64)
plan = C.c_void_p()
assert h.rcg_tiled_plan_create_ex(C.byref(geom), 1, {tile}, {chunk}, {support}, 0,
                                  C.byref(plan)) == 0
n = stub.stub_launches()
assert h.rcg_degrid_tiled_f32(plan, C.byref(gcf), at, at, None) == 0
print(stub.stub_launches() - n)
""")
    assert int(out) == (2 if windows else 3)
