"""FP64 gridding reads one visibility per point: fewer are refused before any
kernel is queued, and of more the first count, with and without a plan (no
GPU: the library's entry points are replaced by a recorder)."""
import numpy as np
import pytest
import torch

from rc_amd import _lib, synth
from rc_amd import device as D
from rc_amd import imaging as IM


class Recorder:
    """Stands for the library: every call is noted and succeeds."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def call(*args):
            self.calls.append((name, args))
            return 0
        return call


@pytest.fixture
def made(monkeypatch):
    rec = Recorder()
    monkeypatch.setattr(_lib, "lib", lambda: rec)
    monkeypatch.setattr(D, "_stream", lambda stream: None)
    vc, gcf, _ = synth.random_small(1, grid_size=64, chunks=4, ts_ch=5)
    geom = D.DeviceGeom.from_chunks(vc, 64, device="cpu")
    dg = D.DeviceGCF.from_table(gcf, device="cpu", dtype=np.complex128)
    return rec, geom, dg


def imager(geom, dg, plan):
    im = object.__new__(IM.Imager)
    im.geom, im.gcf, im.f64, im.cdtype, im.plan = geom, dg, True, torch.complex128, plan
    im.N = im.P = 64
    im.pg = torch.zeros(geom.n * 16, dtype=torch.uint8)
    return im


def plan_of(geom):
    p = object.__new__(D.TiledPlan)
    p.geom, p.n, p.n_inst, p.batch, p._h = geom, geom.n, 1, False, None
    return p


@pytest.mark.parametrize("planned", [False, True])
@pytest.mark.parametrize("n", [0, 19, 20, 21, 40])
def test_visibilities_and_points(made, planned, n):
    rec, geom, dg = made
    assert geom.n == 20
    im = imager(geom, dg, plan_of(geom) if planned else None)
    vis = torch.ones(n, dtype=torch.complex128)
    if n < geom.n:
        with pytest.raises(ValueError):
            im.grid(vis)
        with pytest.raises(ValueError):
            D.grid_plain_f64(geom, dg, im.pg, vis)
        assert not rec.calls
    else:
        im.grid(vis)
        D.grid_plain_f64(geom, dg, im.pg, vis)
        names = [c[0] for c in rec.calls if c[0].startswith("rcg_grid")]
        assert len(names) == 2 and names[1] == "rcg_grid_plain_f64"
        assert names[0].startswith("rcg_grid_tiled_f64" if planned else "rcg_grid_plain_f64")


def test_planned_calls_bring_their_own_counters(made):
    """An Imager is used from several streams: its calls do not share the
    plan's work counters."""
    rec, geom, dg = made
    imager(geom, dg, plan_of(geom)).grid(torch.ones(geom.n, dtype=torch.complex128))
    name, args = [c for c in rec.calls if c[0].startswith("rcg_grid")][0]
    assert name == "rcg_grid_tiled_f64_counters" and args[4] is not None
