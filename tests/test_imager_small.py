"""Whether the FP64 Imager makes a plan: not for so few small windows that
gridding is launches alone (no GPU: the plan is replaced by a recorder)."""
import pytest

from rc_amd import device as D
from rc_amd import imaging as IM
from rc_amd import synth


@pytest.mark.parametrize("chunks,support,option,planned", [
    (1, 4, None, False), (100, 16, None, False), (255, 32, None, False), (256, 32, None, True),
    (1023, 16, None, False), (1024, 16, None, True), (1, 33, None, True), (100, 16, 60, True),
    (4, 33, 8, False)])
def test_plan_or_not(monkeypatch, chunks, support, option, planned):
    made = []

    class Plan:
        def __init__(self, geom, **kw):
            made.append(kw["max_support"])

        def bin(self, gcf):
            pass

        def stats(self):
            return {"err": 0}

    monkeypatch.setattr(D, "TiledPlan", Plan)
    vc, _, _ = synth.random_small(1, grid_size=256, chunks=chunks, ts_ch=1, max_plane=0,
                                  supports=(support,))
    geom = D.DeviceGeom.from_chunks(vc, 256, device="cpu")
    plan = IM.Imager._plan64(geom, None, 32, 512, option)
    assert (plan is not None) == planned
    assert made == ([option or support] if planned else [])
