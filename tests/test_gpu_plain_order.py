"""Plain FP64 degridding adds a window's taps in one order however many points
a call holds: 16 lanes a point (many) sum as a wavefront a point (few) does,
in 64 partial sums, so both give the same bits and neither has the longer
chains' larger rounding errors."""
import numpy as np
import pytest
import torch

from rc_amd import device as D
from rc_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("supports", [(1, 3, 4), (7, 8, 9), (16, 31, 33), (48, 63, 64)])
def test_few_and_many_points_agree(hip_device, supports, half):
    N, n, cut = 200, 6300, 3150
    vc, gcf, _ = synth.random_small(57, grid_size=N, chunks=n, ts_ch=1, half=half,
                                    chunk_supp="random", supports=supports)
    rng = np.random.default_rng(n)
    grid = torch.from_numpy(rng.standard_normal((N, N)) + 1j * rng.standard_normal((N, N))).cuda()
    dg = D.DeviceGCF.from_table(gcf, dtype=np.complex128)

    def degrid(a, b):
        part = synth.VisChunks(uvw=vc.uvw[a:b], vis=vc.vis[a:b], supps=vc.supps[a:b],
                               scale=vc.scale, wstep=vc.wstep)
        geom = D.DeviceGeom.from_chunks(part, N)
        pg, _, err = D.pregrid(geom, dg)
        assert int(err.item()) == 0
        return D.degrid_plain_f64(geom, dg, pg, grid).cpu().numpy().reshape(-1)

    many = degrid(0, n)
    few = np.concatenate([degrid(0, cut), degrid(cut, n)])
    assert np.count_nonzero(many) > n // 2
    assert np.array_equal(many.view(np.uint64), few.view(np.uint64))
