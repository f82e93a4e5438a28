"""The workloads this library is timed on: what its users have it do, through
its public Python entry points.

A case is a dict of plain values; its "kind" names the entry points:

  tiled     device-resident FP32 gridding and degridding: pregrid and tile
            binning of the geometry, gridding of the visibilities and
            degridding of a model grid (rc_amd.device.TiledPlan).  One
            instance, or a batch of instances in one plan.
  operator  one gradient of chi^2 through the differentiable measurement
            operator (rc_amd.operator): forward, and the gridder as backward.
  imager    dirty image of the visibilities and prediction of a model image
            (rc_amd.imaging.Imager), in FP64 (the parity path) or FP32.
  major     the whole major cycle: PSF, dirty image, CLEAN, subtraction.
  ms4       the reference's gridder and degridder entry points on host memory
            (rc_amd.ms4), complex128, chunks of one baseline's samples.
  hogbom    CLEAN minor cycles on a dirty image and its PSF.
  gcf       generation of a w-projection tap table from the points' w.

Points lie as in the synthetic workloads of rc_amd.synth: baselines of a
Gaussian antenna array tracked over hours ("tracks"), the same array's
baselines at random times of a snapshot ("snapshot"), or uniform in the uv
plane with w = 0 ("uniform").  Visibilities are a few point sources plus
noise; taps are a Gaussian envelope times a w-dependent chirp.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from rc_amd import device as D
from rc_amd import gcf as G
from rc_amd import imaging, ms4
from rc_amd import operator as OP
from rc_amd.tables import OVER, GCFTable, VisChunks

WAVELENGTH = 299792458.0 / 1.4e9


def listed() -> list[dict]:
    return [
        # a unit-test sized call, and what a serving loop sends many times:
        # launches and host latency are all there is
        dict(name="tiled_tiny", kind="tiled", layout="tracks", points=612, times=18, grid=256,
             pitch=256, planes=4, s_min=8, s_max=14, half=True, ts=1, zoom=1.0, inst=1,
             tile=32, chunk=512),
        # plain convolutional gridding without w: 512^2, 100 chunks of 1000
        # points, one 8 x 8 kernel
        dict(name="tiled_plain_512", kind="tiled", layout="uniform", points=100000, times=1000,
             grid=512, pitch=512, planes=1, s_min=8, s_max=8, half=False, ts=1000, zoom=1.0,
             inst=1, tile=32, chunk=512),
        # ragged: a side that no tile divides, padded rows, odd supports, a
        # full (signed-plane) table, per-baseline chunk supports that cut
        # windows, and some baselines outside the grid
        dict(name="tiled_ragged_600", kind="tiled", layout="tracks", points=306000, times=306,
             grid=600, pitch=613, planes=9, s_min=7, s_max=31, half=False, ts=306, zoom=1.15,
             inst=1, tile=32, chunk=512),
        # the benchmark's own workload: 4096^2, 32 w-planes, 9,987,840 points
        dict(name="tiled_wproj_4096", kind="tiled", layout="tracks", points=9987840, times=306,
             grid=4096, pitch=4096, planes=32, s_min=8, s_max=64, half=True, ts=1, zoom=1.0,
             inst=1, tile=32, chunk=1024),
        # a batch of uneven snapshots, one launch per stage over all of them
        dict(name="tiled_batch_2048", kind="tiled", layout="snapshot", points=400000, times=1,
             grid=2048, pitch=2048, planes=16, s_min=8, s_max=48, half=True, ts=1, zoom=1.0,
             inst=16, tile=32, chunk=1024),
        # an iterative reconstruction's inner step
        dict(name="operator_2048", kind="operator", layout="tracks", points=4993920, times=153,
             grid=2048, pitch=2048, planes=16, s_min=8, s_max=48, half=True, ts=1, zoom=1.0),
        # imaging at the reference's precision
        dict(name="imager_f64_1024", kind="imager", f64=True, layout="tracks", points=500310,
             times=153, grid=1024, pitch=1024, planes=8, s_min=8, s_max=24, half=True, ts=1,
             zoom=1.0),
        # a whole imaging run of a small field
        dict(name="major_1024", kind="major", f64=False, layout="tracks", points=500310,
             times=153, grid=1024, pitch=1024, planes=8, s_min=8, s_max=24, half=True, ts=1,
             zoom=1.0, majors=2, niters=100),
        # the reference's own calls on host memory: the plain configuration
        # and a w-projection observation
        dict(name="ms4_plain_512", kind="ms4", layout="uniform", points=100000, times=1000,
             grid=512, pitch=512, planes=1, s_min=8, s_max=8, half=False, ts=1000, zoom=1.0),
        dict(name="ms4_wproj_2048", kind="ms4", layout="tracks", points=2496960, times=306,
             grid=2048, pitch=2048, planes=16, s_min=8, s_max=48, half=True, ts=306, zoom=1.0),
        # the deconvolution of a full dirty image
        dict(name="hogbom_2048", kind="hogbom", f64=False, grid=2048, pitch=2048, niters=1000,
             points=1000000, times=306),
        # the tap table of an observation: planes -31..31, supports 8..64
        dict(name="gcf_63_planes", kind="gcf", layout="tracks", points=999906, times=306,
             w_planes=31, s_min=8, growth=2, s_max=64, theta=0.1),
    ]


def _log(rng, lo, hi) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choices(["tiled", "operator", "imager", "major", "ms4", "hogbom", "gcf"],
                       [5, 1, 1, 1, 2, 1, 1])[0]
    grid = _log(rng, 96, 1024) * 2
    if kind == "hogbom":
        return dict(kind=kind, f64=rng.random() < 0.25, grid=grid,
                    pitch=grid + rng.choice([0, 0, 4, 13]), niters=_log(rng, 20, 1000),
                    points=_log(rng, 2000, 1000000), times=rng.choice([60, 153, 306]))
    if kind == "gcf":
        half = rng.randint(2, 31)
        s_min = rng.choice([8, 8, 9, 12, 15])
        return dict(kind=kind, layout="tracks", points=_log(rng, 1000, 2000000),
                    times=rng.choice([60, 153, 306]), w_planes=half, s_min=s_min,
                    growth=rng.choice([1, 2]), s_max=rng.choice([24, 32, 48, 64]),
                    theta=rng.choice([0.02, 0.05, 0.1]))
    s_min = rng.choice([4, 6, 8, 8, 8, 9, 11])
    s_max = s_min + 2 * rng.randint(0, min(28, (grid // 3 - s_min) // 2))
    c = dict(kind=kind, layout=rng.choice(["tracks", "tracks", "snapshot"]),
             points=_log(rng, 500, 3000000), times=rng.choice([18, 60, 153, 306]), grid=grid,
             pitch=grid, planes=rng.randint(2, 32) if s_max > s_min else 1, s_min=s_min,
             s_max=s_max, half=rng.random() < 0.6, ts=1, zoom=rng.choice([1.0, 1.0, 1.1]))
    if c["planes"] == 1 and rng.random() < 0.5:
        c["layout"] = "uniform"
    if c["layout"] == "tracks" and (kind == "ms4" or rng.random() < 0.4):
        c["ts"] = c["times"]
    elif kind == "ms4":
        c["ts"] = rng.choice([1, 50, 1000])
    if kind == "operator":
        c["half"] = True
    elif kind in ("tiled", "ms4") and rng.random() < 0.3:
        c["pitch"] = grid + rng.choice([4, 13, 32])
    if kind == "imager":
        c["f64"] = rng.random() < 0.6
        c["points"] = min(c["points"], 1000000)
    if kind == "major":
        c["f64"] = rng.random() < 0.3
        c["points"] = min(c["points"], 1000000)
        c["majors"] = rng.randint(1, 3)
        c["niters"] = _log(rng, 10, 200)
    if kind == "tiled":
        c["inst"] = rng.choice([1, 1, 1, 2, 5, 9])
        c["points"] = max(500, c["points"] // c["inst"])
        c["tile"] = 32
        c["chunk"] = rng.choice([512, 512, 1024])
    return c


# ---------------------------------------------------------------------------
# inputs


def _gen(seed: int, device) -> torch.Generator:
    g = torch.Generator(device=device)
    g.manual_seed(int(seed))
    return g


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device=g.device, dtype=torch.float64)


def _uniform(g, lo, hi, *shape):
    return lo + (hi - lo) * torch.rand(*shape, generator=g, device=g.device, dtype=torch.float64)


def _baselines(g, n_bl):
    """(X, Y, Z) wavelengths of n_bl antenna pairs of a 256-antenna Gaussian
    array (sigma 800 m, within 3 km): the first n_bl pairs of all."""
    ant = _normal(g, 256, 2) * 800.0
    r = torch.hypot(ant[:, 0], ant[:, 1])
    ant *= torch.where(r > 3000.0, 3000.0 / r, torch.ones_like(r))[:, None]
    lat = math.radians(-30.7)
    i, j = torch.triu_indices(256, 256, 1, device=g.device)
    pick = torch.randperm(i.numel(), generator=g, device=g.device)
    pick = pick.repeat(-(-n_bl // pick.numel()))[:n_bl]
    if n_bl == i.numel():
        pick = torch.arange(n_bl, device=g.device)
    d = (ant[j[pick]] - ant[i[pick]]) / WAVELENGTH
    return -math.sin(lat) * d[:, 1], d[:, 0], math.cos(lat) * d[:, 1]


def _rotate_earth(b, H):
    """uvw of baselines (X, Y, Z) at hour angles H, declination -45."""
    X, Y, Z = b
    dec = math.radians(-45.0)
    s, c = torch.sin(H), torch.cos(H)
    u = s * X + c * Y
    v = -math.sin(dec) * c * X + math.sin(dec) * s * Y + math.cos(dec) * Z
    w = math.cos(dec) * c * X - math.cos(dec) * s * Y + math.sin(dec) * Z
    return torch.stack([u, v, w], -1)


def _uvw(case, g, n):
    """uvw [n, 3] of one instance and the pixel scale-free (w) extent."""
    hour = math.pi / 12.0
    if case.get("layout") == "uniform":
        lim = case["grid"] / 2 - 1 - case["s_max"] / 2
        uvw = torch.zeros(n, 3, dtype=torch.float64, device=g.device)
        uvw[:, :2] = _uniform(g, -lim, lim, n, 2)
        return uvw
    t = case["times"]
    if case.get("layout") == "snapshot":
        b = _baselines(g, n)
        pick = torch.randint(n, (n,), generator=g, device=g.device)
        H = (_uniform(g, -2.0, 2.0, 1) + _uniform(g, -1 / 12, 1 / 12, n)) * hour
        return _rotate_earth([x[pick] for x in b], H)
    n_bl = -(-n // t)
    b = [x[:, None] for x in _baselines(g, n_bl)]
    H = torch.linspace(-2.0, 2.0, t, dtype=torch.float64, device=g.device) * hour
    return _rotate_earth(b, H[None, :]).reshape(-1, 3)[:n].contiguous()


def _counts(case, seed) -> list[int]:
    """Points of every instance (uneven in a batch), whole chunks each."""
    ts = case["ts"]
    k = case.get("inst", 1)
    if k == 1:
        f = [1.0]
    else:
        r = np.random.default_rng(1000 + k)
        f = np.clip(np.exp(r.standard_normal(k)), 0.05, 6.0)
    return [max(1, int(case["points"] * x) // ts) * ts for x in f]


def _supports(case) -> list[int]:
    P, a, b = case["planes"], case["s_min"], case["s_max"]
    return [a + (2 * int(round((b - a) / 2 * p / (P - 1))) if P > 1 else 0) for p in range(P)]


class _Obs:
    """One instance's geometry: uvw, chunk supports, scale and w step."""


def _observe(case, g, n) -> _Obs:
    o = _Obs()
    o.uvw = _uvw(case, g, n)
    if case["layout"] == "uniform":
        o.scale, o.wstep = 1.0, 1.0
    else:
        reach = 6000.0 / WAVELENGTH if case["layout"] == "snapshot" else \
            float(o.uvw[:, :2].abs().max())
        o.scale = case["zoom"] * (case["grid"] / 2 - 1 - case["s_max"] / 2) / reach
        top = 6000.0 / WAVELENGTH if case["layout"] == "snapshot" else \
            float(o.uvw[:, 2].abs().max())
        o.wstep = top / max(1, case["planes"] - 1) if case["planes"] > 1 else 4.0 * top
    sup = torch.tensor(_supports(case), dtype=torch.int32, device=g.device)
    plane = torch.round(o.uvw[:, 2].abs() / o.wstep).long().clamp_(max=case["planes"] - 1)
    o.supps = sup[plane].view(-1, case["ts"]).amin(1).contiguous()
    return o


def _taps(case, dtype, device):
    """Taps of all layers in table order (a full table's planes -M..M, a half
    one's 0..M): Gaussian envelope (sigma S/6) times exp(i pi p r^2 / S^2)."""
    out = []
    P = case["planes"]
    for p in (range(P) if case["half"] else range(1 - P, P)):
        S = _supports(case)[abs(p)]
        off = torch.arange(OVER, dtype=torch.float64, device=device)[:, None] / OVER
        x = torch.arange(S, dtype=torch.float64, device=device)[None, :] - S / 2 - off
        k = torch.polar(torch.exp(-x * x * (18.0 / (S * S))), math.pi * p / (S * S) * x * x)
        out.append((k[:, None, :, None] * k[None, :, None, :]).reshape(-1))
    return torch.cat(out).to(dtype)


def _layers(case):
    """(layer_off, layer_len, supps, center, max_w_plane) of that table."""
    P, sup = case["planes"], _supports(case)
    lens = np.repeat([sup[abs(p)] ** 2 for p in (range(P) if case["half"] else range(1 - P, P))],
                     OVER * OVER)
    offs = np.concatenate([[0], np.cumsum(lens)[:-1]])
    supps = np.asarray([sup[abs(p)] for p in range(1 - P, P)], np.int32)
    return (offs.astype(np.int64), lens.astype(np.int32), supps,
            0 if case["half"] else (P - 1) * OVER * OVER, P - 1)


def _device_gcf(case, dtype, device) -> D.DeviceGCF:
    offs, lens, supps, center, M = _layers(case)
    return D.DeviceGCF(data=_taps(case, dtype, device), layer_off=torch.from_numpy(offs).to(device),
                       layer_len=torch.from_numpy(lens).to(device),
                       supps=torch.from_numpy(supps).to(device), center=center, max_w_plane=M,
                       half=case["half"])


def _sources(case, g, k=6):
    """Flux and (l, m) pixel offsets of a few point sources."""
    N = case["grid"]
    flux = torch.exp(0.7 * _normal(g, k)) * 2.0
    lm = torch.randint(-N // 4, N // 4, (k, 2), generator=g, device=g.device).double()
    return flux, lm


def _observed(case, o, g, dtype, noise=0.5):
    """Visibilities of point sources plus noise."""
    flux, lm = _sources(case, g)
    n = o.uvw.shape[0]
    vis = torch.zeros(n, dtype=torch.complex128, device=g.device)
    for f, p in zip(flux.tolist(), lm.tolist()):
        ph = (-2 * math.pi / case["grid"] * o.scale) * (o.uvw[:, 0] * p[0] + o.uvw[:, 1] * p[1])
        vis += torch.polar(torch.full_like(ph, f), ph)
    vis += noise * torch.complex(_normal(g, n), _normal(g, n))
    return vis.to(dtype)


def _model_grid(case, g, dtype, pitch):
    """The uv grid of a few point sources (padding columns zero)."""
    N = case["grid"]
    flux, lm = _sources(case, g)
    x = torch.arange(N, dtype=torch.float64, device=g.device) - N // 2
    a = torch.polar(torch.ones(N, len(flux), dtype=torch.float64, device=g.device),
                    x[:, None] * lm[None, :, 0] * (2 * math.pi / N))
    b = torch.polar(torch.ones(N, len(flux), dtype=torch.float64, device=g.device),
                    x[:, None] * lm[None, :, 1] * (2 * math.pi / N))
    out = torch.zeros(N, pitch, dtype=dtype, device=g.device)
    out[:, :N] = ((a * flux) @ b.T).to(dtype)
    return out


def _sky(case, g, dtype):
    """A model image: a few point sources on a faint background."""
    N, P = case["grid"], case["pitch"]
    flux, lm = _sources(case, g, 20)
    img = torch.zeros(N, P, dtype=dtype, device=g.device)
    img[:, :N] = (1e-3 * _normal(g, N, N)).to(dtype)
    img[(lm[:, 0] + N // 2).long(), (lm[:, 1] + N // 2).long()] += flux.to(dtype)
    return img


def _geom(case, o) -> D.DeviceGeom:
    return D.DeviceGeom(uvw=o.uvw, chunk_supps=o.supps, n_chunks=o.supps.numel(), ts_ch=case["ts"],
                        scale=o.scale, wstep=o.wstep, grid_size=case["grid"],
                        grid_pitch=case["pitch"])


def _dirty(case, g, dtype):
    """Dirty image and PSF of a uniformly weighted observation (nearest-cell
    gridding and an FFT), in rows of the case's pitch."""
    N, P = case["grid"], case["pitch"]
    uvw = _uvw(dict(case, layout="tracks", s_max=8), g, case["points"])
    scale = (N / 2 - 2) / float(uvw[:, :2].abs().max())
    cell = torch.round(uvw[:, :2] * scale).long()
    hit = torch.zeros(N, N, dtype=torch.float64, device=g.device)
    hit[cell[:, 0] + N // 2, cell[:, 1] + N // 2] = 1.0
    hit[N // 2 - cell[:, 0], N // 2 - cell[:, 1]] = 1.0
    hit = torch.fft.ifftshift(hit)
    sky = torch.zeros(N, N, dtype=torch.float64, device=g.device)
    flux, lm = _sources(case, g, 40)
    sky[(lm[:, 0] + N // 2).long(), (lm[:, 1] + N // 2).long()] += flux
    noise = 0.02 * _normal(g, N, N)
    norm = N * N / float(hit.sum())
    psf = torch.fft.fftshift(torch.fft.ifft2(hit).real) * norm
    res = torch.fft.ifft2(hit * torch.fft.fft2(sky + noise)).real * norm
    out = []
    for img in (res, psf):
        p = torch.zeros(N, P, dtype=dtype, device=g.device)
        p[:, :N] = img.to(dtype)
        out.append(p)
    return out


# ---------------------------------------------------------------------------
# one pass


class _State:
    pass


def _inputs(case, seed, device):
    """The numerical inputs of a case (no plan, no library call)."""
    s = _State()
    s.case = case
    g = _gen(seed, device)
    kind = case["kind"]
    if kind == "hogbom":
        s.res, s.psf = _dirty(case, g, torch.float64 if case["f64"] else torch.float32)
        return s
    if kind == "gcf":
        s.uvw = _uvw(dict(case, grid=1024), g, case["points"])
        s.wstep = float(s.uvw[:, 2].abs().max()) / case["w_planes"]
        return s
    f64 = kind == "ms4" or case.get("f64", False)
    dtype = torch.complex128 if f64 else torch.complex64
    s.obs = [_observe(case, g, n) for n in _counts(case, seed)]
    if len(s.obs) > 1:  # the instances of a plan share the table and its w step
        top = max(o.wstep for o in s.obs)
        sup = torch.tensor(_supports(case), dtype=torch.int32, device=device)
        for o in s.obs:
            o.wstep = top
            plane = torch.round(o.uvw[:, 2].abs() / top).long().clamp_(max=case["planes"] - 1)
            o.supps = sup[plane].view(-1, case["ts"]).amin(1).contiguous()
    noise = 0.05 if kind == "major" else 0.5
    s.vis = torch.cat([_observed(case, o, g, dtype, noise) for o in s.obs])
    if kind in ("tiled", "ms4"):
        s.grid = torch.stack([_model_grid(case, g, dtype, case["pitch"]) for _ in s.obs])
        if case.get("inst", 1) == 1:
            s.grid = s.grid[0]
    elif kind in ("operator", "imager"):
        s.sky = _sky(case, g, torch.float64 if f64 else torch.float32)
    return s


def prepare(case, seed):
    s = _inputs(case, seed, "cuda")
    kind = case["kind"]
    if kind in ("hogbom", "gcf"):
        return s
    if kind == "ms4":
        o = s.obs[0]
        offs, lens, supps, center, M = _layers(case)
        s.table = GCFTable(data=_taps(case, torch.complex128, "cuda").cpu().numpy(),
                           layer_off=offs, layer_len=lens, center=center, supps=supps,
                           max_w_plane=M, half=case["half"])
        nc = o.supps.numel()
        s.chunks = VisChunks(uvw=o.uvw.cpu().numpy().reshape(nc, case["ts"], 3),
                             vis=s.vis.cpu().numpy().reshape(nc, case["ts"]),
                             supps=o.supps.cpu().numpy(), scale=o.scale, wstep=o.wstep)
        s.grid = s.grid.cpu().numpy()
        # the caller's output arrays, as a driver that reuses them holds them
        s.grid_out = np.zeros_like(s.grid)
        s.vis_out = np.zeros_like(s.chunks.vis)
        s.grid_out[...] = 1.0
        s.vis_out[...] = 1.0
        return s
    f64 = case.get("f64", False)
    s.gcf = _device_gcf(case, torch.complex128 if f64 else torch.complex64, "cuda")
    geoms = [_geom(case, o) for o in s.obs]
    if kind == "tiled":
        s.plan = D.TiledPlan(geoms if case["inst"] > 1 else geoms[0], tile=case["tile"],
                             chunk=case["chunk"], max_support=case["s_max"])
    elif kind == "operator":
        s.op = OP.MeasurementOp(geoms[0], s.gcf, max_support=case["s_max"])
    else:
        s.im = imaging.Imager(geoms[0], s.gcf, f64=f64, max_support=case["s_max"])
    return s


def run(s):
    case = s.case
    kind = case["kind"]
    if kind == "tiled":
        s.plan.bin(s.gcf)
        return {"grid": s.plan.grid(s.gcf, s.vis), "vis": s.plan.degrid(s.gcf, s.grid)}
    if kind == "operator":
        x = s.sky.detach().requires_grad_(True)
        OP.chi2(s.op, x, s.vis).backward()
        return {"grad": x.grad}
    if kind == "imager":
        return {"dirty": s.im.image(s.vis), "vis": s.im.predict(s.sky)}
    if kind == "major":
        r = s.im.major_cycles(s.vis, case["majors"], case["niters"], 0.1, 0.0)
        return {k: r[k] for k in ("residual", "model", "vis", "psf")}
    if kind == "ms4":
        N, P = case["grid"], case["pitch"]
        g, taps = ms4.grid(s.chunks, s.table, N, P, out=s.grid_out)
        v, taps2 = ms4.degrid(s.chunks, s.table, s.grid, N, out=s.vis_out)
        return {"grid": g, "vis": v, "taps": taps, "degrid_taps": taps2}
    if kind == "hogbom":
        res = s.res.clone()
        model, iters = D.hogbom(res, s.psf, case["niters"], 0.1, 0.0)
        return {"residual": res, "model": model, "iters": iters}
    table, info = G.make_gcf(s.uvw, s.wstep, case["theta"], case["s_min"], case["growth"],
                             case["s_max"], max_w_plane=case["w_planes"])
    return {"taps": table.data, "means": [float(x) for x in info["means"]][:60],
            "npts": np.asarray(info["npts"])}


# ---------------------------------------------------------------------------
# what a pass cannot do without


def work(case):
    kind = case["kind"]
    N, P = case.get("grid", 0), case.get("pitch", 0)
    if kind == "hogbom":
        b = 8 if case["f64"] else 4
        # residual and PSF read, residual and model written; one multiply and
        # one subtraction per pixel and component
        return {"bytes": 4.0 * b * N * N, "flops": 2.0 * N * N * case["niters"]}
    if kind == "gcf":
        sup = [min(case["s_max"], case["s_min"] + case["growth"] * abs(p))
               for p in range(-case["w_planes"], case["w_planes"] + 1)]
        L, ms = OVER * case["s_max"], case["s_max"]
        # a separable transform of the ms^2 screen to each window's samples
        fl = sum(8.0 * (OVER * S * ms * ms + (OVER * S) ** 2 * ms) for S in sup)
        return {"bytes": 24.0 * case["points"] + 8.0 * 64 * sum(S * S for S in sup),
                "flops": min(fl, len(sup) * 10.0 * L * L * math.log2(L))}
    g = _gen(1, "cpu")
    sample = dict(case, points=max(case["ts"], 20000 // case["ts"] * case["ts"]), inst=1)
    o = _observe(sample, g, sample["points"])
    mean = float((o.supps.double() ** 2).mean())
    n = float(sum(_counts(case, 0)))
    taps = n * mean
    f64 = kind == "ms4" or case.get("f64", False)
    b = 16.0 if f64 else 8.0
    inst = case.get("inst", 1)
    table = b * float(_layers(case)[1].sum())
    grid = b * N * P * inst
    points = (24.0 + b) * n
    fft = 5.0 * N * N * math.log2(N * N)
    one = points + table + grid
    if kind in ("tiled", "ms4"):
        return {"bytes": 2 * one, "flops": 16 * taps}
    if kind == "operator":
        return {"bytes": 2 * one + 8.0 * n + 8.0 * N * N, "flops": 16 * taps + 2 * fft}
    if kind == "imager":
        return {"bytes": 2 * one + b * N * N, "flops": 16 * taps + 1.5 * fft}
    k = case["majors"]
    return {"bytes": 2 * k * one, "flops": 8 * taps * 2 * k + 1.5 * k * fft +
            2.0 * N * N * case["niters"] * k}


# ---------------------------------------------------------------------------
# 64-bit values by plain torch


def _windows(case, o):
    """Of the in-bound points: their index, first cell, first tap, row stride,
    window side and whether their taps are conjugated."""
    N = case["grid"]
    offs, lens, supps, center, M = (torch.from_numpy(x).to(o.uvw.device)
                                    if isinstance(x, np.ndarray) else x for x in _layers(case))
    S = o.supps.long().repeat_interleave(case["ts"])
    us, vs = o.uvw[:, 0] * o.scale, o.uvw[:, 1] * o.scale
    fu, fv = torch.floor(us), torch.floor(vs)
    ou, ov = torch.floor(8 * (us - fu)).long(), torch.floor(8 * (vs - fv)).long()
    q = o.uvw[:, 2] / o.wstep
    t = torch.trunc(q)
    wp = (t + torch.where((q - t).abs() >= 0.5, torch.sign(q), torch.zeros_like(q))).long()
    u0 = fu.long() + N // 2 - torch.div(S, 2, rounding_mode="trunc")
    v0 = fv.long() + N // 2 - torch.div(S, 2, rounding_mode="trunc")
    ok = (u0 >= 0) & (u0 < N - S) & (v0 >= 0) & (v0 < N - S)
    slot = (wp.abs() if case["half"] else wp) * 64 + ou * 8 + ov + center
    gs = supps.long()[(wp + M).clamp(0, 2 * M)]
    tap0 = offs[slot.clamp(0, offs.numel() - 1)] + (gs - S) // 2 * (gs + 1)
    i = torch.nonzero(ok).flatten()
    return (i, (u0 * case["pitch"] + v0)[i], tap0[i], gs[i], S[i],
            ((wp < 0) if case["half"] else torch.zeros_like(ok))[i])


def _each_row(case, o, taps, conj_all=False):
    """(points, cells, taps) of every window row, all windows of one side and
    at most 8 M taps at a time."""
    idx, cell, tap0, stride, S, conj = _windows(case, o)
    conj = conj ^ conj_all
    for side in torch.unique(S).tolist():
        of_side = torch.nonzero(S == side).flatten()
        for p in torch.split(of_side, max(1, (8 << 20) // side)):
            col = torch.arange(side, device=p.device)
            c0, t0, st = cell[p][:, None] + col, tap0[p][:, None] + col, stride[p][:, None]
            sign = torch.where(conj[p], -1.0, 1.0).double()[:, None]
            for r in range(side):
                t = taps[t0 + r * st]
                yield idx[p], c0 + r * case["pitch"], torch.complex(t.real, t.imag * sign)


def _grid64(case, o, taps, vis, conj_all=False):
    size = case["grid"] * case["pitch"]
    re = torch.zeros(size, dtype=torch.float64, device=vis.device)
    im = torch.zeros_like(re)
    for i, c, t in _each_row(case, o, taps, conj_all):
        x = vis[i][:, None] * t
        re.index_add_(0, c.reshape(-1), x.real.reshape(-1))
        im.index_add_(0, c.reshape(-1), x.imag.reshape(-1))
    return torch.complex(re, im).view(case["grid"], case["pitch"])


def _degrid64(case, o, taps, grid):
    out = torch.zeros(o.uvw.shape[0], dtype=torch.complex128, device=grid.device)
    g = grid.reshape(-1)
    for i, c, t in _each_row(case, o, taps):
        out[i] += (g[c] * t).sum(1)
    return out


def _fft(x, sign):
    f = torch.fft.fft2 if sign < 0 else torch.fft.ifft2
    y = torch.fft.fftshift(f(torch.fft.fftshift(x)))
    return y if sign < 0 else y * x.numel()


def _dirty64(case, o, taps, vis):
    """Grid, normalise, fold the upper half onto the lower, half-complex to
    real transform."""
    N, P = case["grid"], case["pitch"]
    g = _grid64(case, o, taps, vis)[:, :N] / float(N * P)
    fold = g.clone()
    fold[:, :N // 2] += g.flip(0, 1)[:, :N // 2].conj()
    half = torch.fft.fftshift(fold)[:, :N // 2 + 1]
    img = torch.fft.irfft2(half, s=(N, N)) * (N * N)
    return torch.fft.fftshift(img)


def _predict64(case, o, taps, img):
    g = torch.zeros(case["grid"], case["pitch"], dtype=torch.complex128, device=img.device)
    g[:, :case["grid"]] = _fft(img.to(torch.complex128), -1)
    return _degrid64(case, o, taps, g)


def _clean64(res, psf, niters, gain):
    N = res.shape[0]
    model = torch.zeros_like(res)
    p = int(psf.abs().argmax())
    pr, pc = divmod(p, N)
    top = float(psf[pr, pc])
    for _ in range(niters):
        r, c = divmod(int(res.abs().argmax()), N)
        a = gain * float(res[r, c]) / top
        r0, r1, c0, c1 = max(0, r - pr), min(N, N + r - pr), max(0, c - pc), min(N, N + c - pc)
        res[r0:r1, c0:c1] -= a * psf[r0 - r + pr:r1 - r + pr, c0 - c + pc:c1 - c + pc]
        model[r, c] += a
    return model


def _layer64(case, S, w):
    """One plane's [8, 8, S, S] taps: the w screen on an s_max^2 block, its
    zero-padded transform sampled by two matrix products, each sub-lattice
    divided by its own sum of real parts."""
    ms = case["s_max"]
    L, R = OVER * ms, ms // 2
    i = torch.arange(-R, R + ms % 2, dtype=torch.float64, device="cuda")
    x = i * (case["theta"] / 2 / R)
    ph = w * case["theta"] * (1 - torch.sqrt(1 - x[:, None] ** 2 - x[None, :] ** 2))
    screen = torch.polar(torch.ones_like(ph), -2 * math.pi * ph)
    k = torch.arange(L, dtype=torch.float64, device="cuda") - L // 2
    a = (2 * math.pi / L) * torch.remainder(k[:, None] * i[None, :], float(L))
    E = torch.polar(torch.ones_like(a), a)
    full = E @ screen @ E.T
    sums = full.real.reshape(ms, OVER, ms, OVER).sum((0, 2))
    st = (ms // 2 - S // 2) * OVER
    sub = full[st:st + S * OVER, st:st + S * OVER].reshape(S, OVER, S, OVER)
    return (sub.permute(1, 3, 0, 2) / sums[:, :, None, None]).reshape(-1)


def exact(case, seed):
    kind = case["kind"]
    s = _inputs(case, seed, "cuda")
    if kind == "hogbom":
        N = case["grid"]
        res, psf = s.res[:, :N].double(), s.psf[:, :N].double()
        model = _clean64(res, psf, case["niters"], 0.1)
        out = []
        for img in (res, model):
            p = torch.zeros(N, case["pitch"], dtype=torch.float64, device="cuda")
            p[:, :N] = img
            out.append(p)
        return {"residual": out[0], "model": out[1], "iters": None}
    if kind == "gcf":
        M = case["w_planes"]
        w = s.uvw[:, 2]
        q = w / s.wstep
        t = torch.trunc(q)
        plane = (t + torch.where((q - t).abs() >= 0.5, torch.sign(q),
                                 torch.zeros_like(q))).long() + M
        sums = torch.zeros(2 * M + 1, dtype=torch.float64, device="cuda").index_add_(0, plane, w)
        npts = torch.bincount(plane, minlength=2 * M + 1)
        means = [float(sums[k] / npts[k]) if npts[k] else s.wstep * (k - M)
                 for k in range(2 * M + 1)]
        taps = [_layer64(case, min(case["s_max"], case["s_min"] + case["growth"] * abs(k - M)),
                         means[k]) for k in range(2 * M + 1)]
        return {"taps": torch.cat(taps), "means": means[:60], "npts": None}
    f64 = kind == "ms4" or case.get("f64", False)
    o = s.obs[0]
    # the taps as the call sees them, in 64 bits
    taps = _taps(case, torch.complex128 if f64 else torch.complex64, "cuda").to(torch.complex128)
    vis = s.vis.to(torch.complex128)
    if kind in ("tiled", "ms4"):
        grids, out, at = [], [], 0
        models = s.grid if s.grid.dim() == 3 else s.grid[None]
        for k, o in enumerate(s.obs):
            n = o.uvw.shape[0]
            grids.append(_grid64(case, o, taps, vis[at:at + n]))
            out.append(_degrid64(case, o, taps, models[k].to(torch.complex128)))
            at += n
        if kind == "ms4":
            return {"grid": grids[0].cpu().numpy(), "vis": out[0].view(-1, case["ts"]).cpu().numpy(),
                    "taps": None, "degrid_taps": None}
        return {"grid": torch.stack(grids) if len(grids) > 1 else grids[0], "vis": torch.cat(out)}
    if kind == "operator":
        r = _predict64(case, o, taps, s.sky.double()) - vis
        return {"grad": _fft(_grid64(case, o, taps, 2 * r, conj_all=True), 1).real}
    if kind == "imager":
        return {"dirty": _dirty64(case, o, taps, vis),
                "vis": _predict64(case, o, taps, s.sky.double())}
    psf = _dirty64(case, o, taps, torch.ones_like(vis))
    total = torch.zeros_like(psf)
    for k in range(case["majors"]):
        res = _dirty64(case, o, taps, vis)
        model = _clean64(res, psf, case["niters"], 0.1)
        total += model
        if k + 1 < case["majors"]:
            vis = vis - _predict64(case, o, taps, model)
    return {"residual": res, "model": total, "vis": vis, "psf": psf}
