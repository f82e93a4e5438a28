"""GCF layers by matrix products against the numpy oracle at the block edges:
rows in blocks of 32, columns in blocks of 16, terms four at a time, several
planes per launch, tables whose screen does not fit in LDS.  Bar as in
test_gpu_gcf: 1e-12 of the largest tap."""
import numpy as np
import pytest
import torch

from oracle import gcf_oracle as G
from rc_amd import _lib
from rc_amd import gcf as GG

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("max_support,supports", [
    (2, [1, 2]), (3, [1, 2, 3]), (15, [3, 15, 4]), (16, [16, 4, 5]), (17, [17, 2]),
    (33, [33, 31]), (64, [64, 63]), (130, [6, 130]), (150, [7]), (158, [4]), (241, [2]), (256, [3]),
    (6, [1 + k % 6 for k in range(67)])])  # two launches
def test_layers_vs_oracle(hip_device, max_support, supports):
    t2 = 0.03
    w = np.linspace(-90.0, 120.0, len(supports))
    sizes = [64 * s * s for s in supports]
    offs = np.concatenate([[0], np.cumsum(sizes)])[:-1]
    gen = GG.GCFGenerator(max_support, 4)
    dst = torch.full((int(sum(sizes)) + 5,), 7.0, dtype=torch.complex128, device="cuda")
    gen.layers(dst, supports, offs, t2, w)
    got = dst.cpu().numpy()
    gen.close()
    assert (got[-5:] == 7.0).all()
    for k, s in enumerate(supports):
        exp = G.mk_gcf_layer(s, max_support, 0, t2, float(w[k]))
        have = got[offs[k]:offs[k] + sizes[k]].reshape(8, 8, s, s)
        assert np.abs(have - exp).max() <= 1e-12 * np.abs(exp).max()


def test_generator_keeps_shutdown_refused(hip_device):
    gen = GG.GCFGenerator(8, 0)
    assert _lib.lib().rcg_shutdown() != 0
    gen.close()
