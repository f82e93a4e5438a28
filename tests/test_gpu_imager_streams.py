"""FP64 gridding through one Imager on several streams and threads at once:
the calls share the plan, each with work counters of its own.  Every result
equals the plain gridder's to FP64 rounding."""
import threading

import numpy as np
import pytest
import torch

from rc_amd import device as D
from rc_amd import imaging as IM
from rc_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("threads", [1, 4])
def test_streams_share_an_imager(hip_device, threads):
    vc, gcf, _ = synth.wproj(seed=9, n_ant=60, n_times=20, grid_size=256, n_planes=4, s_min=8,
                             s_max=16, vis_dtype=np.complex128)
    geom = D.DeviceGeom.from_chunks(vc, 256)
    dg = D.DeviceGCF.from_table(gcf, dtype=np.complex128)
    im = IM.Imager(geom, dg, f64=True, chunk=64)
    assert im.plan is not None and im.plan.stats()["items"] > 300
    vis = [torch.from_numpy(vc.vis.reshape(-1) * (k + 1.5j)).cuda() for k in range(4)]
    ref = [D.grid_plain_f64(geom, dg, im.pg, v) for v in vis]
    streams = [torch.cuda.Stream() for _ in vis]
    torch.cuda.synchronize()
    bad = []

    def work(mine):
        try:
            for _ in range(12):
                outs = []
                for k in mine:
                    with torch.cuda.stream(streams[k]):
                        outs.append((k, im.grid(vis[k])))
                for k, g in outs:
                    streams[k].synchronize()
                    err = float((g - ref[k]).abs().max() / ref[k].abs().max())
                    if err > 1e-13:
                        bad.append((k, err))
        except Exception as e:  # noqa: BLE001
            bad.append(e)

    ts = [threading.Thread(target=work, args=(range(k, 4, threads),)) for k in range(threads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
    im.close()
