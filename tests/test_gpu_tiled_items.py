"""GPU parity of the tiled FP32 path over its work-item table and queues: the
numbers of items per tile at which the table's writer and the queues' ranges
change.  Bars as in test_gpu_tiled: relative L2 <= 1e-5 against the FP64
oracle on complex64-rounded inputs."""
import numpy as np
import pytest

from conftest import rel_l2
from oracle import oracle as O
from rc_amd import synth
from test_gpu_tiled import TOL, c64_round, run_tiled

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", ["pairs", "halo"])
@pytest.mark.parametrize("n,chunk,items", [(1, 1, 1), (7, 2, 4), (9, 2, 5), (64, 1, 64),
                                           (65, 1, 65), (4099, 1, 4099)])
def test_items_of_one_tile_vs_oracle(hip_device, layout, n, chunk, items):
    """All windows in one 32x32 tile, cut into 1, 4, 5 (the lane writes up to
    4), 64, 65 (a wavefront's width) and 4099 items (more than the workgroups
    that own a first item; ranges of unequal length)."""
    vc, gcf, _ = synth.random_small(31, grid_size=160, chunks=n, ts_ch=1, half=True,
                                    supports=(6, 8, 10), oob_frac=0.0)
    rng = np.random.default_rng(n)
    # first cells 65..86 for u, v in [-10, 10]: every window in cells 64..95
    vc.uvw[:, 0, :2] = rng.uniform(-10.0, 10.0, (n, 2)) / vc.scale
    vc, gcf = c64_round(vc, gcf)
    ref, taps = O.grid(vc, gcf, 160, nthreads=4)
    ref32 = ref.astype(np.complex64).astype(np.complex128)
    vref, _ = O.degrid(vc, gcf, ref32, nthreads=4)
    g, v, st = run_tiled(vc, gcf, 160, 32, chunk, grid_in=ref32, layout=layout)
    assert st["err"] == 0 and st["taps"] == taps and st["items"] == items
    assert rel_l2(g, ref) <= TOL
    assert rel_l2(v, vref) <= TOL
