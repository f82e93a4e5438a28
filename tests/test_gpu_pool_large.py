"""MS4 calls whose arrays are copied by several threads through pinned
buffers (8 MiB and more to the device, 3 MiB and more back), from several
host threads at once.  Every result equals the oracle's (FP64, 1e-12)."""
import threading

import numpy as np
import pytest

from conftest import rel_l2
from oracle import oracle as O
from rc_amd import ms4, synth

pytestmark = pytest.mark.gpu


def test_staged_copies_from_several_threads(hip_device):
    cases = []
    for k, (N, chunks) in enumerate([(512, 530), (600, 360), (460, 700)]):
        vc, gcf, _ = synth.random_small(70 + k, grid_size=N, chunks=chunks, ts_ch=1000,
                                        half=k % 2 == 1, supports=(4, 5, 6))
        assert vc.uvw.nbytes >= 8 << 20 and 16 * N * N >= 3 << 20
        ref, taps = O.grid(vc, gcf, N, nthreads=8)
        vref, _ = O.degrid(vc, gcf, ref, nthreads=8)
        cases.append((vc, gcf, N, ref, taps, vref))
    assert any(c[0].vis.nbytes >= 8 << 20 for c in cases)
    bad = []

    def work(c):
        vc, gcf, N, ref, taps, vref = c
        try:
            for _ in range(4):
                g, n = ms4.grid(vc, gcf, N)
                assert n == taps and rel_l2(g, ref) <= 1e-12
                v, n = ms4.degrid(vc, gcf, ref, N)
                assert n == taps and rel_l2(v, vref) <= 1e-12
        except Exception as e:  # noqa: BLE001
            bad.append(e)

    ts = [threading.Thread(target=work, args=(c,)) for c in cases * 2]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
