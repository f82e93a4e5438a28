"""The pad_quirk arena of a GCF generator, over a stand-in for the HIP runtime
(no GPU): made with the generator, so that no call allocates and any may be
captured, or on first use where that was asked for."""
import hipstub


def test_arena_comes_with_the_generator(tmp_path):
    out = hipstub.run(tmp_path, """
g = C.c_void_p()
dst = C.create_string_buffer(64 * 8 * 8 * 16)
def layer(quirk):
    n = stub.stub_launches()
    assert h.rcg_gcf_gen_layer(g, C.addressof(dst), 1, 8, 0.1, 3.0, quirk, None) == 0
    assert stub.stub_launches() > n
arena = (8 * 32) * (8 * 32 + 4) * 16
assert h.rcg_gcf_gen_create(32, 4, C.byref(g)) == 0
made = stub.stub_live()
assert made >= arena
for quirk in (1, 0, 1):
    layer(quirk)
    assert stub.stub_live() == made
h.rcg_gcf_gen_destroy(g)
assert stub.stub_live() == 0
stub.stub_limit(arena - 1)
assert h.rcg_gcf_gen_create(32, 4, C.byref(g)) == 3 and not g.value   # RCG_ERR_NOMEM
assert stub.stub_live() == 0
assert h.rcg_gcf_gen_create_ex(32, 4, 0, C.byref(g)) == 0
layer(0)
assert stub.stub_live() == 0
stub.stub_limit(1 << 30)
layer(1)
assert stub.stub_live() == made
h.rcg_gcf_gen_destroy(g)
assert stub.stub_live() == 0 and h.rcg_shutdown() == 0
print("ok")
""")
    assert out.split() == ["ok"]
