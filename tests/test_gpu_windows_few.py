"""Degridding by whole windows where tiles hold few points (a wavefront per
point) and many (staged regions), in one plan: against the FP64 oracle on
complex64-rounded inputs, relative L2 <= 1e-5, and bit for bit the same after
binning again."""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from oracle import oracle as O
from rc_amd import device as D
from rc_amd import synth
from test_gpu_tiled import TOL, c64_round

pytestmark = pytest.mark.gpu


def scattered(seed, N, supports, dense, sparse, half=True, cs="random"):
    """`dense` points in two tiles' worth of cells and `sparse` over the grid."""
    vc, gcf, _ = synth.random_small(seed, grid_size=N, chunks=dense + sparse, ts_ch=1, half=half,
                                    chunk_supp=cs, supports=supports, oob_frac=0.0)
    rng = np.random.default_rng(seed)
    edge = N / 2 - max(supports) // 2 - 2
    p = rng.uniform(-edge, edge, (dense + sparse, 2))
    p[:dense] = rng.uniform(-16.0, 16.0, (dense, 2))
    vc.uvw[:, 0, :2] = p / vc.scale
    return c64_round(vc, gcf)


def plan_of(vc, gcf, N, pitch, tile, chunk):
    geom = D.DeviceGeom.from_chunks(vc, N, pitch)
    dg = D.DeviceGCF.from_table(gcf, dtype=np.complex64)
    plan = D.TiledPlan(geom, tile=tile, chunk=chunk)
    plan.bin(dg)
    assert plan.stats()["err"] == 0
    return plan, dg


@pytest.mark.parametrize("tile,supports", [(16, (1, 9, 48)), (32, (1, 2, 3)), (32, (8, 17, 63)),
                                           (32, (16, 31, 64)), (64, (5, 8, 31))])
@pytest.mark.parametrize("dense,sparse", [(0, 1), (0, 7), (0, 400), (1500, 300)])
def test_few_and_many_vs_oracle(hip_device, tile, supports, dense, sparse):
    N = 500
    vc, gcf = scattered(71 + sparse, N, supports, dense, sparse)
    rng = np.random.default_rng(4)
    gin = rng.standard_normal((N, N + 5)) + 1j * rng.standard_normal((N, N + 5))
    gin = gin.astype(np.complex64)
    want, taps = O.degrid(vc, gcf, gin.astype(np.complex128), size=N, nthreads=4)
    plan, dg = plan_of(vc, gcf, N, N + 5, tile, 512)
    assert plan.stats()["taps"] == taps > 0
    g = torch.from_numpy(gin).cuda()
    first = plan.degrid(dg, g).cpu().numpy()
    assert rel_l2(first.reshape(want.shape), want) <= TOL
    assert np.array_equal(first.reshape(want.shape) == 0, want == 0)
    for _ in range(3):
        plan.bin(dg)
        assert np.array_equal(plan.degrid(dg, g).cpu().numpy(), first)
    plan.close()


def test_nan_stays_outside_the_window(hip_device):
    """A NaN cell reaches exactly the points whose window holds it, of tiles
    with few points and with many."""
    N = 300
    vc, gcf = scattered(83, N, (6, 9, 17), 900, 120)
    gin = np.ones((N, N), np.complex64)
    gin[70::9, 66::11] = np.nan
    want, _ = O.degrid(vc, gcf, gin.astype(np.complex128), nthreads=4)
    plan, dg = plan_of(vc, gcf, N, N, 32, 512)
    got = plan.degrid(dg, torch.from_numpy(gin).cuda()).cpu().numpy().reshape(want.shape)
    plan.close()
    hit = np.isnan(want.real)
    assert hit.any() and not hit.all() and np.array_equal(np.isnan(got.real), hit)
    assert rel_l2(got[~hit], want[~hit]) <= TOL


def test_batch_of_dense_and_sparse_instances(hip_device):
    """Instances of 3, 2000 and 40 points in one plan."""
    N, parts = 260, []
    for k, (dense, sparse) in enumerate([(0, 3), (1900, 100), (0, 40)]):
        parts.append(scattered(90 + k, N, (7, 8, 30), dense, sparse))
    gcf = parts[0][1]
    vcs = [p[0] for p in parts]
    rng = np.random.default_rng(5)
    gin = rng.standard_normal((3, N, N)) + 1j * rng.standard_normal((3, N, N))
    gin = gin.astype(np.complex64)
    dg = D.DeviceGCF.from_table(gcf, dtype=np.complex64)
    plan = D.TiledPlan([D.DeviceGeom.from_chunks(vc, N) for vc in vcs], tile=32, chunk=512)
    plan.bin(dg)
    got = plan.degrid(dg, torch.from_numpy(gin).cuda()).cpu().numpy()
    plan.close()
    at = 0
    for vc, g in zip(vcs, gin):
        want, _ = O.degrid(vc, gcf, g.astype(np.complex128), nthreads=4)
        n = want.size
        assert rel_l2(got[at:at + n].reshape(want.shape), want) <= TOL
        at += n


def test_time_of_sparse_points(hip_device):
    """20,000 points of 48 x 48 spread over 4096^2, about one a tile: at most
    two and a half times as long as by pairs, which a plan of small items
    takes (165 against 100 us; staging a region for every point took 445)."""
    n, N, S = 20000, 4096, 48
    g = torch.Generator("cuda")
    g.manual_seed(3)
    uvw = torch.zeros(n, 3, dtype=torch.float64, device="cuda")
    uvw[:, :2] = (torch.rand(n, 2, generator=g, device="cuda", dtype=torch.float64) - 0.5) * 3900
    k = torch.arange(64, device="cuda")
    gcf = D.DeviceGCF(data=torch.randn(64 * S * S, generator=g, device="cuda").to(torch.complex64),
                      layer_off=k * (S * S),
                      layer_len=torch.full((64,), S * S, dtype=torch.int32, device="cuda"),
                      supps=torch.tensor([S], dtype=torch.int32, device="cuda"), center=0,
                      max_w_plane=0, half=True)
    geom = D.DeviceGeom(uvw=uvw, chunk_supps=torch.full((n,), S, dtype=torch.int32, device="cuda"),
                        n_chunks=n, ts_ch=1, scale=1.0, wstep=1.0, grid_size=N, grid_pitch=N)
    grid = torch.ones(N, N, dtype=torch.complex64, device="cuda")
    t = {}
    for chunk in (512, 128):
        plan = D.TiledPlan(geom, tile=32, chunk=chunk)
        plan.bin(gcf)
        plan.timing(True)
        for _ in range(10):
            plan.degrid(gcf, grid)
        t[chunk] = min(plan.kernel_times("degrid"))
        plan.close()
    assert t[512] <= 2.5 * t[128]
