"""Hogbom CLEAN on tiles against whole-image passes in numpy with the same
arithmetic (the component's amplitude rounded to the image's type, one product
and one subtraction per pixel, in order): residual, model and iteration count
are equal bit for bit."""
import numpy as np
import pytest
import torch

from rc_amd import device as D

pytestmark = pytest.mark.gpu


def passes(res, psf, siz, niters, gain, threshold):
    res, psf = res.copy(), psf[:, :siz]
    model = np.zeros_like(res)
    p = int(np.argmax(np.abs(psf)))
    pr, pc = divmod(p, siz)
    pval = float(psf[pr, pc])
    it = 0
    for it in range(niters + 1):
        if it == niters:
            break
        x = res[:, :siz]
        r, c = divmod(int(np.argmax(np.abs(x))), siz)
        v = float(x[r, c])
        if abs(v) < threshold or pval == 0.0:
            break
        a = res.dtype.type(gain * v / pval)
        r0, r1 = max(0, r - pr), min(siz, siz + r - pr)
        c0, c1 = max(0, c - pc), min(siz, siz + c - pc)
        res[r0:r1, c0:c1] -= a * psf[r0 - r + pr:r1 - r + pr, c0 - c + pc:c1 - c + pc]
        model[r, c] += a
    return res, model, it


def sky(rng, siz, pitch, dtype, noise):
    """Residual and PSF: a few sources through a beam with far sidelobes."""
    k = np.fft.fftfreq(siz)
    mask = (rng.random((siz, siz)) < 0.3) & (np.hypot(k[:, None], k[None, :]) < 0.4)
    mask |= np.roll(mask[::-1, ::-1], 1, (0, 1))
    mask[0, 0] = True  # never empty: a 1 x 1 image has this sample only
    beam = np.fft.ifft2(mask).real
    beam /= beam[0, 0]
    img = np.zeros((siz, siz))
    for _ in range(6):
        img[rng.integers(siz), rng.integers(siz)] += rng.uniform(0.5, 2.0) * rng.choice([-1, 1])
    img += noise * rng.standard_normal((siz, siz))
    dirty = np.fft.ifft2(np.fft.fft2(beam) * np.fft.fft2(img)).real
    out = []
    for x in (dirty, np.fft.fftshift(beam)):
        y = np.full((siz, pitch), 7.0, dtype)  # columns past the image are not part of it
        y[:, :siz] = x
        out.append(y)
    return out


def run(res, psf, niters, gain, threshold):
    r = torch.from_numpy(res).cuda()
    model, it = D.hogbom(r, torch.from_numpy(psf).cuda(), niters, gain, threshold)
    return r.cpu().numpy(), model.cpu().numpy(), it


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("siz,pitch,niters,noise", [
    (1, 1, 3, 1.0), (31, 31, 40, 0.1),    # one tile, partial
    (32, 35, 16, 0.05),                   # one tile, one round of iterations
    (65, 70, 17, 0.3),                    # three tiles a side, one iteration in a second round
    (64, 64, 129, 0.3),
    (200, 200, 300, 0.02),
    (200, 213, 300, 1.0),                 # noise: many tiles near the peak
    (530, 530, 260, 0.3)])                # 17 tiles a side
def test_tiles_equal_passes(hip_device, dtype, siz, pitch, niters, noise):
    rng = np.random.default_rng(siz + niters)
    res, psf = sky(rng, siz, pitch, dtype, noise)
    want, wmodel, wit = passes(res, psf, siz, niters, 0.1, 0.0)
    got, model, it = run(res, psf, niters, 0.1, 0.0)
    assert it == wit
    assert np.array_equal(got, want)
    assert np.array_equal(model, wmodel)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_tiles_above_2048(hip_device, dtype):
    """2112^2: tiles of 64 pixels a side."""
    rng = np.random.default_rng(9)
    res, psf = sky(rng, 2112, 2120, dtype, 0.01)
    want, wmodel, wit = passes(res, psf, 2112, 20, 0.1, 0.0)
    got, model, it = run(res, psf, 20, 0.1, 0.0)
    assert it == wit and np.array_equal(got, want) and np.array_equal(model, wmodel)


def test_threshold_ties_and_flat_images(hip_device):
    """The threshold stops in the middle of a round; equal maxima in many
    tiles (more than are visited at a time) are taken first index first; a
    zero image and a zero PSF leave everything as it was."""
    rng = np.random.default_rng(5)
    res, psf = sky(rng, 160, 160, np.float32, 0.01)
    want, wmodel, wit = passes(res, psf, 160, 400, 0.2, 0.5)
    got, model, it = run(res, psf, 400, 0.2, 0.5)
    assert 0 < wit < 400 and it == wit
    assert np.array_equal(got, want) and np.array_equal(model, wmodel)
    siz = 640  # 400 tiles
    flat = np.where(rng.random((siz, siz)) < 0.5, -1.0, 1.0).astype(np.float32)
    delta = np.zeros((siz, siz), np.float32)
    delta[300, 310], delta[300, 311] = 1.0, -1.0  # equal PSF peaks: the first
    want, wmodel, wit = passes(flat, delta, siz, 150, 0.5, 0.0)
    got, model, it = run(flat, delta, 150, 0.5, 0.0)
    assert it == wit and np.array_equal(got, want) and np.array_equal(model, wmodel)
    for res, psf in ((np.zeros_like(flat), delta), (flat, np.zeros_like(delta))):
        got, model, it = run(res, psf, 5, 0.1, 1e-3)
        assert it == 0 and np.array_equal(got, res) and not model.any()
