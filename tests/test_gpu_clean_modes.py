"""CLEAN on tiles and by passes over the whole image: where the work goes over
from one to the other, with one threshold, NaNs and infinities among the
pixels, and an image on which the pruning of tiles finds nothing to prune.
Residual, model and iteration count equal whole-image passes in numpy bit for
bit; rcg_hogbom (passes only) and rcg_hogbom_run agree."""
import ctypes as C

import numpy as np
import pytest
import torch

from rc_amd import _lib
from rc_amd import device as D
from test_gpu_clean_tiles import passes, sky

pytestmark = pytest.mark.gpu


def run(name, res, psf, siz, niters, gain, threshold):
    """(residual, model, iterations, whether passes took over)"""
    h = _lib.lib()
    r, p = torch.from_numpy(res).cuda(), torch.from_numpy(psf).cuda()
    m = torch.full_like(r, 5.0)
    scratch = torch.zeros(int(h.rcg_hogbom_scratch_bytes()), dtype=torch.uint8, device="cuda")
    args = (m.data_ptr(), r.data_ptr(), p.data_ptr(), int(res.dtype == np.float64), siz,
            res.shape[1], niters, gain, threshold, scratch.data_ptr())
    s = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    it = C.c_uint(99)
    if name == "rcg_hogbom_run":
        _lib.check(h.rcg_hogbom_run(*args, C.byref(it), s), name)
    else:
        _lib.check(h.rcg_hogbom(*args, s), name)
        _lib.check(h.rcg_hogbom_iterations(scratch.data_ptr(), C.byref(it), s), name)
    over = int(scratch[40:44].view(torch.int32).item())  # CleanState::passes
    return r.cpu().numpy(), m.cpu().numpy(), it.value, over


def snapshot(rng, siz, pitch, dtype, points):
    """A few sources seen by a short observation: sidelobes of tens of per
    cent over the whole field."""
    hit = np.zeros((siz, siz))
    k = np.clip(np.rint(rng.standard_normal((points, 2)) * siz * 0.13), 1 - siz // 2,
                siz // 2 - 1).astype(int)
    hit[k[:, 0], k[:, 1]] = 1.0
    hit[-k[:, 0], -k[:, 1]] = 1.0
    img = np.zeros((siz, siz))
    img[rng.integers(siz, size=20), rng.integers(siz, size=20)] += rng.uniform(0.5, 2.0, 20)
    beam = np.fft.ifft2(hit).real * siz * siz / hit.sum()
    out = []
    for x in (np.fft.ifft2(np.fft.fft2(img) * np.fft.fft2(beam)).real, np.fft.fftshift(beam)):
        y = np.full((siz, pitch), 7.0, dtype)
        y[:, :siz] = x
        out.append(y)
    return out


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("siz,pitch,niters,kind,over", [
    (399, 399, 70, "dense", 0),       # below the size from which tiles are tried
    (400, 403, 1, "dense", 0), (400, 400, 16, "dense", 0), (430, 437, 250, "dense", None),
    (513, 520, 17, "snapshot", None),
    (700, 700, 200, "snapshot", 1),   # over in mid-run
    (640, 640, 40, "flat", 1)])       # over in the first iteration
def test_both_ways_equal_numpy(hip_device, dtype, siz, pitch, niters, kind, over):
    rng = np.random.default_rng(siz)
    if kind == "dense":
        res, psf = sky(rng, siz, pitch, dtype, 0.02)
    elif kind == "snapshot":
        res, psf = snapshot(rng, siz, pitch, dtype, 60)
    else:
        res = np.where(rng.random((siz, pitch)) < 0.5, -1.0, 1.0).astype(dtype)
        psf = np.zeros((siz, pitch), dtype)
        psf[siz // 2, siz // 2:siz // 2 + 2] = 1.0, -0.25
    for threshold in (0.0, None):
        if threshold is None:  # stops half way
            if niters < 16:
                continue
            threshold = 0.5 * (abs(first) + abs(last))
        want, wmodel, wit = passes(res, psf, siz, niters, 0.1, threshold)
        if threshold == 0.0:
            first, last = np.abs(res[:, :siz]).max(), np.abs(want[:, :siz]).max()
        for name in ("rcg_hogbom_run", "rcg_hogbom"):
            got, model, it, went = run(name, res, psf, siz, niters, 0.1, threshold)
            assert it == wit
            assert np.array_equal(got, want) and np.array_equal(model[:, :siz], wmodel[:, :siz])
            if name == "rcg_hogbom_run" and threshold == 0.0 and over is not None:
                assert went == over


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_nan_and_inf_pixels(hip_device, dtype):
    """A NaN pixel is never a peak and an infinite one always; the subtraction
    of an infinite component leaves infinities and NaNs.  Images of NaNs, and a
    PSF of NaNs, stop at once."""
    siz = 450
    rng = np.random.default_rng(4)
    res, psf = sky(rng, siz, siz, dtype, 0.02)
    res[5, 7] = res[200:260, 100:300] = np.nan
    r = np.where(np.isnan(res), 0, res)
    want, wmodel, wit = passes(r, psf, siz, 60, 0.1, 0.0)
    nan = np.isnan(res)
    for name in ("rcg_hogbom_run", "rcg_hogbom"):
        got, model, it, _ = run(name, res, psf, siz, 20, 0.1, 0.0)
        assert it == 20 and np.array_equal(np.isnan(got), nan) and not np.isnan(model).any()
    a = run("rcg_hogbom_run", res, psf, siz, 60, 0.1, 0.0)
    b = run("rcg_hogbom", res, psf, siz, 60, 0.1, 0.0)
    assert all(np.array_equal(x, y, equal_nan=True) for x, y in zip(a[:3], b[:3]))
    res[300, 300] = np.inf
    a = run("rcg_hogbom_run", res, psf, siz, 40, 0.1, 0.0)
    b = run("rcg_hogbom", res, psf, siz, 40, 0.1, 0.0)
    assert np.isinf(a[1][300, 300]) and a[2] == b[2]
    assert all(np.array_equal(x, y, equal_nan=True) for x, y in zip(a[:2], b[:2]))
    for x, y in ((np.full_like(res, np.nan), psf), (np.nan_to_num(r), np.full_like(psf, np.nan))):
        for name in ("rcg_hogbom_run", "rcg_hogbom"):
            got, model, it, _ = run(name, x, y, siz, 10, 0.1, 0.0)
            assert it == 0 and np.array_equal(got, x, equal_nan=True) and not model.any()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_time_does_not_hang_on_the_image(hip_device, dtype):
    """1024^2, an iteration on a zero image (every tile can hold the peak) and
    on noise with a PSF of one pixel (few can): at most five times as long."""
    siz = 1024
    psf = torch.zeros(siz, siz, dtype=dtype, device="cuda")
    psf[siz // 2, siz // 2] = 1.0
    g = torch.Generator("cuda")
    g.manual_seed(1)
    noise = torch.randn(siz, siz, generator=g, device="cuda", dtype=torch.float64).to(dtype)

    def best(img):
        out = []
        for _ in range(4):
            r = img.clone()
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            D.hogbom(r, psf, 96, 0.1, 0.0)
            b.record()
            b.synchronize()
            out.append(a.elapsed_time(b))
        return min(out)

    assert best(torch.zeros_like(noise)) <= 5.0 * best(noise)
