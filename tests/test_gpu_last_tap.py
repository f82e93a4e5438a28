"""Degridding by whole windows with the very last tap of the table: odd,
uncut windows of the last layer (offset (7, 7) of the last plane), whose
16-byte load straddles the table's end.  That tap outweighs all others, so a
point that loses it is off by far.  Bar: 1e-5 per point against the FP64
oracle on complex64-rounded inputs."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from rc_amd import device as D
from rc_amd import synth
from test_gpu_tiled import TOL, c64_round

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("S", [1, 3, 9, 31, 63])
def test_last_tap(hip_device, half, S):
    N = 200
    vc, gcf, _ = synth.random_small(61, grid_size=N, chunks=60, ts_ch=1, max_plane=2, half=half,
                                    supports=(8, 6, S), oob_frac=0.0)
    rng = np.random.default_rng(S)
    cell = rng.integers(-30, 30, (60, 2)) + 0.9375  # over-sampling offset 7
    vc.uvw[:, 0, :2] = cell / vc.scale
    vc.uvw[:, 0, 2] = 2 * vc.wstep
    vc.supps[:] = S
    gcf.data[-1] = 40.0 * S * S
    vc, gcf = c64_round(vc, gcf)
    gin = (rng.standard_normal((N, N)) + 1j * rng.standard_normal((N, N)))
    gin = gin.astype(np.complex64)
    want, taps = O.degrid(vc, gcf, gin.astype(np.complex128), nthreads=2)
    assert taps == 60 * S * S
    dg = D.DeviceGCF.from_table(gcf, dtype=np.complex64)
    plan = D.TiledPlan(D.DeviceGeom.from_chunks(vc, N), tile=32, chunk=512, max_support=S)
    plan.bin(dg)
    got = plan.degrid(dg, torch.from_numpy(gin).cuda()).cpu().numpy().reshape(want.shape)
    plan.close()
    assert (np.abs(got - want) <= TOL * np.abs(want).max()).all()
    # (without that tap every point would be another)
    gcf.data[-1] = 0.0
    without, _ = O.degrid(vc, gcf, gin.astype(np.complex128), nthreads=2)
    assert (np.abs(without - want) > 100 * TOL * np.abs(want).max()).mean() > 0.9
