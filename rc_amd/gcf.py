"""GCF tables generated on the device (librcgrid.so rcg_gcf_* / rcg_calc_accums).

make_gcf() follows the reference's GCF kernel (MS4/dna-programs/Kernel/CPU/
GCF.hs:36-89): per-plane supports min(max_size, min_size + growth*|p|) for
planes -M..M, the mean w of every plane's points (or the plane's nominal w
when it has none), and one mkGCFLayer per plane with w = mean * theta and
t2 = theta / 2.  The result is a full (signed-plane) table ready for the
gridders.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import torch

from . import _lib
from .device import DeviceGCF, _stream
from .tables import OVER


class GCFGenerator(_lib.Handle):
    """rcg_gcf_gen for one max_support/src_pad.  arena: with the FP64 arena and
    rocFFT plan that pad_quirk needs; without, its first use makes them."""

    def __init__(self, max_support: int, src_pad: int = 4, arena: bool = True):
        h = C.c_void_p()
        _lib.check(_lib.lib().rcg_gcf_gen_create_ex(max_support, src_pad, int(arena),
                                                    C.byref(h)), "rcg_gcf_gen_create")
        self.max_support, self.src_pad = max_support, src_pad
        self._own(h)

    def layer(self, dst: torch.Tensor, support: int, t2: float, w: float,
              pad_quirk: bool = False, stream=None) -> torch.Tensor:
        """One plane's 64 layers [8, 8, support, support] into dst
        (complex128 or complex64, contiguous, 64*support^2 elements)."""
        if dst.numel() != OVER * OVER * support * support or not dst.is_contiguous():
            raise ValueError("dst must hold 64*support^2 contiguous elements")
        f64 = dst.dtype == torch.complex128
        if not f64 and dst.dtype != torch.complex64:
            raise TypeError("dst must be complex128 or complex64")
        _lib.check(_lib.lib().rcg_gcf_gen_layer(self._h, dst.data_ptr(), int(f64), support,
                                                t2, w, int(pad_quirk), _stream(stream)),
                   "rcg_gcf_gen_layer")
        return dst

    def layers(self, dst: torch.Tensor, supports, offsets, t2: float, w, pad_quirk: bool = False,
               stream=None) -> torch.Tensor:
        """The layers of several planes into dst (complex128 or complex64,
        contiguous): plane k's, of supports[k] for phase w[k], from element
        offsets[k] on; one launch for up to 64 planes."""
        f64 = dst.dtype == torch.complex128
        if not f64 and dst.dtype != torch.complex64:
            raise TypeError("dst must be complex128 or complex64")
        sup = np.ascontiguousarray(supports, np.int32)
        off = np.ascontiguousarray(offsets, np.int64)
        ws = np.ascontiguousarray(w, np.float64)
        if not dst.is_contiguous() or not len(sup) == len(off) == len(ws) or \
                (len(sup) and int((off + 64 * sup.astype(np.int64) ** 2).max()) > dst.numel()):
            raise ValueError("dst must hold every plane's 64*support^2 contiguous elements")
        _lib.check(_lib.lib().rcg_gcf_gen_layers(self._h, dst.data_ptr(), int(f64), len(sup),
                                                 sup.ctypes.data, off.ctypes.data, t2,
                                                 ws.ctypes.data, int(pad_quirk),
                                                 _stream(stream)), "rcg_gcf_gen_layers")
        return dst

    DESTROY = "rcg_gcf_gen_destroy"


def _accums(uvw: torch.Tensor, wstep: float, n_planes: int, stream):
    """calc_accums's results as views of one byte tensor (and that tensor)."""
    uvw = uvw.reshape(-1, 3)
    if uvw.dtype != torch.float64 or not uvw.is_contiguous():
        raise TypeError("uvw must be contiguous float64 [n, 3]")
    buf = torch.empty(12 * n_planes + 4, dtype=torch.uint8, device=uvw.device)
    sums = buf[:8 * n_planes].view(torch.float64)
    npts = buf[8 * n_planes:12 * n_planes].view(torch.int32)
    err = buf[12 * n_planes:].view(torch.int32)
    _lib.check(_lib.lib().rcg_calc_accums(uvw.data_ptr(), uvw.shape[0], wstep, n_planes,
                                          sums.data_ptr(), npts.data_ptr(), err.data_ptr(),
                                          _stream(stream)), "rcg_calc_accums")
    return sums, npts, err, buf


def calc_accums(uvw: torch.Tensor, wstep: float, n_planes: int,
                stream=None) -> tuple[torch.Tensor, torch.Tensor, int]:
    """Per-plane sum of w and point count (device tensors), and the error
    word (bit 0: points outside the planes, skipped)."""
    sums, npts, err, _ = _accums(uvw, wstep, n_planes, stream)
    return sums, npts, int(err.item())


def make_gcf(uvw: torch.Tensor, wstep: float, theta: float, min_size: int, growth: int,
             max_size: int, max_w_plane: int | None = None, src_pad: int = 4,
             pad_quirk: bool = False, dtype=torch.complex64, stream=None
             ) -> tuple[DeviceGCF, dict]:
    """Full GCF table for planes -M..M on the device; returns the table and
    {"supps", "means", "npts"} (host lists)."""
    uvw = uvw.reshape(-1, 3)
    if max_w_plane is None:
        w = uvw[:, 2]
        max_w_plane = max(int(torch.round(w.max() / wstep).item()),
                          int(torch.round(-w.min() / wstep).item()), 0)
    M = int(max_w_plane)
    n_planes = 2 * M + 1
    host = _accums(uvw, wstep, n_planes, stream)[3].cpu().numpy()  # one copy
    sums = host[:8 * n_planes].view(np.float64)
    npts = host[8 * n_planes:12 * n_planes].view(np.int32)
    if int(host[12 * n_planes:].view(np.int32)[0]):
        raise _lib.RcgError("make_gcf: points outside the w-planes")
    supps = [min(max_size, min_size + growth * abs(p)) for p in range(-M, M + 1)]
    means = []
    wmid = -wstep * M
    for k in range(n_planes):
        means.append(sums[k] / npts[k] if npts[k] > 0 else wmid)
        wmid = wmid + wstep
    sup = np.asarray(supps, np.int64)
    lens = np.repeat(sup * sup, OVER * OVER)
    offs = np.concatenate([[0], np.cumsum(lens)])
    dev = uvw.device
    data = torch.empty(int(offs[-1]), dtype=dtype, device=dev)
    # (the arena and its plan take milliseconds to make)
    gen = GCFGenerator(max_size, src_pad, arena=pad_quirk)
    try:
        gen.layers(data, sup, offs[:-1:OVER * OVER], theta / 2.0, np.asarray(means) * theta,
                   pad_quirk, stream)
        # offsets, lengths and supports in one copy
        n = len(lens)
        idx = np.empty(12 * n + 4 * n_planes, np.uint8)
        idx[:8 * n].view(np.int64)[:] = offs[:-1]
        idx[8 * n:12 * n].view(np.int32)[:] = lens
        idx[12 * n:].view(np.int32)[:] = sup
        idx = torch.from_numpy(idx).to(dev)
        torch.cuda.current_stream().synchronize() if stream is None else stream.synchronize()
    finally:
        gen.close()
    table = DeviceGCF(data=data, layer_off=idx[:8 * n].view(torch.int64),
                      layer_len=idx[8 * n:12 * n].view(torch.int32),
                      supps=idx[12 * n:].view(torch.int32), center=M * OVER * OVER, max_w_plane=M,
                      half=False)
    return table, {"supps": supps, "means": means, "npts": npts.tolist()}
