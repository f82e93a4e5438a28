"""The MS4 calls on device memory kept from earlier calls: alternating sizes,
a call after one that failed, several threads at once, and after the kept
memory was given back.  Every result equals the oracle's (FP64, 1e-12)."""
import threading

import numpy as np
import pytest

from conftest import rel_l2
from oracle import oracle as O
from rc_amd import _lib, ms4, synth
from rc_amd.tables import GCFTable, VisChunks

pytestmark = pytest.mark.gpu


def case(seed, N, chunks):
    vc, gcf, _ = synth.random_small(seed, grid_size=N, chunks=chunks, ts_ch=11, half=seed % 2 == 1,
                                    supports=(6, 9, 16))
    ref, taps = O.grid(vc, gcf, N, nthreads=2)
    vref, _ = O.degrid(vc, gcf, ref, nthreads=2)
    return vc, gcf, N, ref, taps, vref


def check(c):
    vc, gcf, N, ref, taps, vref = c
    g, n = ms4.grid(vc, gcf, N)
    assert n == taps and rel_l2(g, ref) <= 1e-12
    v, n = ms4.degrid(vc, gcf, ref, N)
    assert n == taps and rel_l2(v, vref) <= 1e-12


def test_sizes_errors_and_trim(hip_device):
    cs = [case(1, 96, 20), case(2, 300, 400), case(3, 97, 21), case(4, 64, 1)]
    for c in cs + cs[::-1]:
        check(c)
    vc, gcf, N = cs[1][:3]
    # a chunk support above its plane's: refused, with work already queued
    bad = VisChunks(uvw=vc.uvw, vis=vc.vis, supps=np.full_like(vc.supps, 20), scale=vc.scale,
                    wstep=vc.wstep)
    with pytest.raises(_lib.RcgError):
        ms4.grid(bad, gcf, N)
    for c in cs:
        check(c)
    _lib.lib().rcg_shutdown()  # gives the kept memory back
    for c in cs:
        check(c)


def test_layers_apart_in_memory(hip_device):
    """Layers that do not follow each other are gathered; a table that starts
    with unused planes is read from where its used ones begin."""
    c = case(5, 96, 20)
    vc, gcf, N, ref, taps, vref = c
    gap = 7
    data = np.zeros(len(gcf.data) + gap * gcf.n_slots, np.complex128)
    off = gcf.layer_off + gap * np.arange(gcf.n_slots)
    for o, p, n in zip(gcf.layer_off, off, gcf.layer_len):
        data[p:p + n] = gcf.data[o:o + n]
    apart = GCFTable(data=data, layer_off=off, layer_len=gcf.layer_len, center=gcf.center,
                     supps=gcf.supps, max_w_plane=gcf.max_w_plane, half=gcf.half)
    check((vc, apart, N, ref, taps, vref))
    vc.uvw[..., 2] = 0.0  # plane 0 only, whose support is 6
    vc.supps[:] = 6
    ref, taps = O.grid(vc, gcf, N, nthreads=2)
    vref, _ = O.degrid(vc, gcf, ref, nthreads=2)
    check((vc, gcf, N, ref, taps, vref))


def test_threads(hip_device):
    cs = [case(10 + k, 80 + 31 * k, 15 + 9 * k) for k in range(6)]
    bad = []

    def work(c):
        try:
            for _ in range(8):
                check(c)
        except Exception as e:  # noqa: BLE001
            bad.append(e)

    ts = [threading.Thread(target=work, args=(c,)) for c in cs]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
