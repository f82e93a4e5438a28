"""One plane of a large support takes no longer by matrix products than by the
whole transform that pad_quirk runs on the same generator (half as long again
is allowed for), and its taps are the oracle's to 1e-12 of the largest."""
import numpy as np
import pytest
import torch

from oracle import gcf_oracle as G
from rc_amd import gcf as GG

pytestmark = pytest.mark.gpu


def best_ms(f, n=8, inner=5):
    f()
    out = []
    for _ in range(n):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        for _ in range(inner):
            f()
        b.record()
        b.synchronize()
        out.append(a.elapsed_time(b) / inner)
    return min(out)


@pytest.mark.parametrize("ms", [128, 129, 256])
def test_single_layer_time(hip_device, ms):
    gen = GG.GCFGenerator(ms, 4)
    dst = torch.empty(64 * ms * ms, dtype=torch.complex128, device="cuda")
    whole = best_ms(lambda: gen.layer(dst, ms, 0.05, 90.0, pad_quirk=True))
    one = best_ms(lambda: gen.layer(dst, ms, 0.05, 90.0))
    gen.close()
    assert one <= 1.5 * whole


@pytest.mark.parametrize("ms,S", [(97, 97), (98, 96), (191, 20), (192, 33), (255, 6), (256, 9)])
def test_large_layers_vs_oracle(hip_device, ms, S):
    gen = GG.GCFGenerator(ms, 0)
    dst = torch.empty(64 * S * S, dtype=torch.complex128, device="cuda")
    have = gen.layer(dst, S, 0.04, -77.0).cpu().numpy().reshape(8, 8, S, S)
    gen.close()
    exp = G.mk_gcf_layer(S, ms, 0, 0.04, -77.0)
    assert np.abs(have - exp).max() <= 1e-12 * np.abs(exp).max()
