"""The FP64 Imager with and without a plan: options that no plan takes (they
were ignored before) still work, and both gridders agree to FP64 rounding."""
import numpy as np
import pytest
import torch

from rc_amd import device as D
from rc_amd import imaging as IM
from rc_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("opts,planned", [({}, True), ({"tile": 16, "chunk": 3}, True),
                                          ({"tile": 7}, False), ({"chunk": 0}, False),
                                          ({"max_support": 1}, False)])
def test_fp64_imager_plan_or_not(hip_device, opts, planned):
    vc, gcf, _ = synth.wproj(seed=6, n_ant=20, n_times=20, grid_size=128, n_planes=4, s_min=8,
                             s_max=16, vis_dtype=np.complex128)
    geom = D.DeviceGeom.from_chunks(vc, 128, 132)
    dg = D.DeviceGCF.from_table(gcf, dtype=np.complex128)
    vis = torch.from_numpy(vc.vis.reshape(-1)).cuda()
    pg, taps, _ = D.pregrid(geom, dg)
    ref = D.grid_plain_f64(geom, dg, pg, vis)
    im = IM.Imager(geom, dg, f64=True, **opts)
    assert (im.plan is not None) == planned and im.taps == int(taps.item())
    got = im.grid(vis)
    assert float((got - ref).abs().max()) <= 1e-13 * float(ref.abs().max())
    im.close()
