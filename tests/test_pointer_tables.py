"""The pointer tables of a GCFTable, used by several threads' calls at once:
a later call does not free an earlier one's."""
import ctypes as C

import numpy as np

from rc_amd import synth


def test_tables_of_earlier_calls_stay():
    _, gcf, _ = synth.random_small(3, grid_size=64, chunks=2, ts_ch=2)
    first, supps = gcf.pointer_tables()
    lo = first.value - gcf.center * 8
    want = (gcf.data.ctypes.data + gcf.layer_off * gcf.data.itemsize).astype(np.uint64)
    others = []
    for _ in range(50):  # freed memory of that size would be used again
        gcf.pointer_tables()
        others.append((C.c_void_p * gcf.n_slots)(*[1] * gcf.n_slots))
        others.append(np.full(gcf.supps.size, -1, np.int32))
    got = np.ctypeslib.as_array((C.c_uint64 * gcf.n_slots).from_address(lo))
    assert np.array_equal(got, want)
    M = gcf.max_w_plane
    sup = np.ctypeslib.as_array((C.c_int32 * gcf.supps.size).from_address(supps.value - 4 * M))
    assert np.array_equal(sup, gcf.supps)
