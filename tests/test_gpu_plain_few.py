"""Plain FP64 degridding with a wavefront per point (up to 6144 points) and
with 16 lanes per point: supports around both, cut windows, more points than
one wavefront's, the line between them; and the time of one large window."""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from oracle import oracle as O
from rc_amd import device as D
from rc_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunks", [1, 63, 65, 6143, 6144, 6145])
@pytest.mark.parametrize("supports", [(1, 2, 3), (7, 8, 9), (15, 17, 33)])
def test_vs_oracle(hip_device, chunks, supports):
    N = 120
    vc, gcf, _ = synth.random_small(51, grid_size=N, chunks=chunks, ts_ch=1, half=True,
                                    chunk_supp="random", supports=supports)
    rng = np.random.default_rng(chunks)
    gin = rng.standard_normal((N, N + 3)) + 1j * rng.standard_normal((N, N + 3))
    want, taps = O.degrid(vc, gcf, gin, size=N, nthreads=4)
    geom = D.DeviceGeom.from_chunks(vc, N, N + 3)
    dg = D.DeviceGCF.from_table(gcf, dtype=np.complex128)
    pg, n, err = D.pregrid(geom, dg)
    assert int(err.item()) == 0 and int(n.item()) == taps
    got = D.degrid_plain_f64(geom, dg, pg, torch.from_numpy(gin).cuda()).cpu().numpy()
    if np.any(want):
        assert rel_l2(got.reshape(want.shape), want) <= 1e-13
    assert np.array_equal(got.reshape(want.shape) == 0, want == 0)


def best_us(f):
    f()
    out = []
    for _ in range(6):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        for _ in range(10):
            f()
        b.record()
        b.synchronize()
        out.append(a.elapsed_time(b) * 100)
    return min(out)


def test_time_of_one_large_window(hip_device):
    """One point of 256 x 256: 1024 steps of 64 lanes, 4096 of 16.  In units of
    a 16 x 16 window, which is launch and latency alone (7.6 us): 17 with a
    wavefront (129 us), 51 with 16 lanes."""
    t = {}
    for S in (16, 256):
        g = torch.Generator("cuda")
        g.manual_seed(S)
        geom = D.DeviceGeom(uvw=torch.zeros(1, 3, dtype=torch.float64, device="cuda"),
                            chunk_supps=torch.full((1,), S, dtype=torch.int32, device="cuda"),
                            n_chunks=1, ts_ch=1, scale=1.0, wstep=1.0, grid_size=600,
                            grid_pitch=600)
        k = torch.arange(64, device="cuda")
        taps = torch.randn(64 * S * S, generator=g, device="cuda", dtype=torch.float64)
        gcf = D.DeviceGCF(data=taps.to(torch.complex128), layer_off=k * (S * S),
                          layer_len=torch.full((64,), S * S, dtype=torch.int32, device="cuda"),
                          supps=torch.tensor([S], dtype=torch.int32, device="cuda"), center=0,
                          max_w_plane=0, half=True)
        pg, _, _ = D.pregrid(geom, gcf)
        grid = torch.ones(600, 600, dtype=torch.complex128, device="cuda")
        vis = torch.empty(1, dtype=torch.complex128, device="cuda")
        t[S] = best_us(lambda: D.degrid_plain_f64(geom, gcf, pg, grid, vis))
    assert t[256] <= 30 * t[16]
