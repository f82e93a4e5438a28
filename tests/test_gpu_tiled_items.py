"""GPU parity of the tiled FP32 path over its work-item table and queues: the
numbers of items per tile at which the table's writer and the queues' ranges
change.  Bars as in test_gpu_tiled: relative L2 <= 1e-5 against the FP64
oracle on complex64-rounded inputs."""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from oracle import oracle as O
from rc_amd import device as D
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


@pytest.mark.parametrize("tile,supports", [
    (16, (1, 9, 80)), (16, (2, 16, 81)),       # the largest that two workgroups' LDS hold, and
    (32, (1, 17, 64)), (32, (8, 31, 65)),      # one more: whole windows, pairs
    (64, (1, 15, 32)), (64, (3, 16, 33))])
@pytest.mark.parametrize("half,cs", [(False, "random"), (True, "min")])
def test_window_degrid_edges_vs_oracle(hip_device, tile, supports, half, cs):
    """Degridding by whole windows over supports 1, 2, 3 and around 8, 16 and
    32 columns (lanes and steps per row), odd and even ones mixed, truncated
    windows, rows of a padded pitch, tiles that the grid's side cuts, and more
    points per tile than one sort takes."""
    N = 230
    vc, gcf, _ = synth.random_small(41, grid_size=N, chunks=60, ts_ch=40, half=half,
                                    chunk_supp=cs, supports=supports)
    vc, gcf = c64_round(vc, gcf)
    rng = np.random.default_rng(6)
    gin = (rng.standard_normal((N, N + 3)) + 1j * rng.standard_normal((N, N + 3)))
    gin = gin.astype(np.complex64).astype(np.complex128)
    vref, taps = O.degrid(vc, gcf, gin, size=N, nthreads=4)
    _, v, st = run_tiled(vc, gcf, N, tile, 4096, grid_in=gin, pitch=N + 3)
    assert st["err"] == 0 and st["taps"] == taps
    assert rel_l2(v, vref) <= TOL
    assert np.array_equal(v == 0, vref == 0)


def test_window_degrid_keeps_nan_outside_the_window(hip_device):
    """A NaN cell reaches exactly the points whose window holds it: lanes past
    a window's end and an odd window's missing column read neither grid nor
    taps of their neighbours."""
    N = 160
    vc, gcf, _ = synth.random_small(43, grid_size=N, chunks=80, ts_ch=10, half=True,
                                    chunk_supp="random", supports=(6, 9, 17))
    vc, gcf = c64_round(vc, gcf)
    gin = np.ones((N, N), np.complex128)
    gin[70::9, 66::11] = np.nan
    vref, _ = O.degrid(vc, gcf, gin, nthreads=4)
    _, v, st = run_tiled(vc, gcf, N, 32, 64, grid_in=gin)
    assert st["err"] == 0
    hit = np.isnan(vref.real)
    assert hit.any() and not hit.all()
    assert np.array_equal(np.isnan(v.real), hit)
    assert rel_l2(v[~hit], vref[~hit]) <= TOL


def test_window_degrid_above_max_support(hip_device):
    """A support above the plan's max_support whose windows meet no more tiles
    than the plan allows is gridded and degridded as before, without an
    error."""
    vc, gcf, _ = synth.random_small(47, grid_size=160, chunks=70, ts_ch=1, half=True,
                                    supports=(6, 8, 20), oob_frac=0.0)
    rng = np.random.default_rng(8)
    vc.uvw[:, 0, :2] = rng.uniform(-3.0, 3.0, (70, 2)) / vc.scale  # all in cells 64..95
    vc, gcf = c64_round(vc, gcf)
    ref, taps = O.grid(vc, gcf, 160, nthreads=4)
    ref32 = ref.astype(np.complex64)
    vref, _ = O.degrid(vc, gcf, ref32.astype(np.complex128), nthreads=4)
    geom = D.DeviceGeom.from_chunks(vc, 160)
    dg = D.DeviceGCF.from_table(gcf, dtype=np.complex64)
    plan = D.TiledPlan(geom, tile=32, chunk=64, max_support=8)
    plan.bin(dg)
    g = plan.grid(dg, torch.from_numpy(vc.vis.reshape(-1).astype(np.complex64)).cuda())
    v = plan.degrid(dg, torch.from_numpy(ref32).cuda())
    st = plan.stats()
    assert st["err"] == 0 and st["taps"] == taps
    assert rel_l2(g.cpu().numpy(), ref) <= TOL
    assert rel_l2(v.cpu().numpy().reshape(70, 1), vref) <= TOL
    plan.close()


@pytest.mark.parametrize("n,segments", [(512, 1), (528, 2), (2048, 16), (2064, 17), (2160, 18)])
def test_scan_segments_vs_oracle(hip_device, n, segments):
    """Windows over the whole of grids of 1, 2 and 16 segments of 1024 tiles
    (one launch scans them) and of 17 and 18 (three launches), several items
    per tile and a last segment that is not full."""
    assert -(-(-(-n // 16)) ** 2 // 1024) == segments
    vc, gcf, _ = synth.random_small(47, grid_size=n, chunks=500, ts_ch=4, half=True,
                                    supports=(6, 8, 10), oob_frac=0.0)
    rng = np.random.default_rng(n)
    vc.uvw[..., :2] = rng.uniform(-n / 2 + 20, n / 2 - 20, vc.uvw[..., :2].shape) / vc.scale
    vc, gcf = c64_round(vc, gcf)
    ref, taps = O.grid(vc, gcf, n, nthreads=4)
    gin = (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n)))
    gin = gin.astype(np.complex64).astype(np.complex128)
    vref, _ = O.degrid(vc, gcf, gin, nthreads=4)
    g, v, st = run_tiled(vc, gcf, n, 16, 1, grid_in=gin)
    assert st["err"] == 0 and st["taps"] == taps and st["items"] == st["pairs"] > 2000
    assert rel_l2(g, ref) <= TOL
    assert rel_l2(v, vref) <= TOL
