"""The workloads that measure this framework, with float64 results to check them.

``listed()`` names the cases, ``draw(rng)`` gives more of the same ranges,
``prepare`` / ``run`` execute one through the public entry points, and ``exact``
restates it in plain float64 torch.  They stand for what a user has the framework do:

* one tile through the operator interface (``ALGORITHMS[name].process``);
* a whole raster through the tile scheduler (``process_dem``), local and
  spatial mode, float32 / int16 / uint8 output, with and without NoData;
* many independent ragged tiles as one batch (``FusedBatch``), and several
  products of one raster as a captured job (``RasterJob``);
* the learned openness surrogate: inference, and a training step's forward
  and backward passes.

The terrain is seeded spectral fBm, as in the benchmark and the tests; NoData
comes as 1 % discs of radius 5 to 50 px.  File I/O (COG, Zarr) is not among
them: the host's ZSTD and the disk bound it, not this code's kernels.
"""
import math
import os

import numpy as np
import torch

from fujishadergpu_amd import synth
from fujishadergpu_amd.algorithms import ALGORITHMS
from fujishadergpu_amd.batch import FusedBatch, RasterJob, TileJob
from fujishadergpu_amd.scheduler import process_dem
from fujishadergpu_amd.surrogate import Net, WEIGHTS_FILE, surrogate_openness

NODATA = -9999.0
USM_SCALE = 12.5          # a fixed TopoUSM p99 scale (m) where the caller gives one


# ------------------------------------------------------------------- the cases

def listed():
    return [
        # the smallest call: one small tile, where launches and host work count
        dict(name="tile_hillshade_256", kind="tile", algo="hillshade", h=256, w=256, px=10.0,
             nodata=0.0),
        # an ordinary odd-sized tile with NoData holes
        dict(name="tile_curvature_nodata", kind="tile", algo="curvature", h=1000, w=1531,
             px=10.0, nodata=0.01),
        # a raster to int16 with a NoData sentinel, ragged tiles
        dict(name="job_slope_i16_nodata", kind="job", algo="slope", mode="local", h=10007,
             w=8191, px=10.0, nodata=0.01, dtype="int16", tile=4096),
        # the headline: six radii, p99 pre-pass, two output encodings
        dict(name="job_topousm_16384", kind="job", algo="topousm_fast", mode="spatial", h=16384,
             w=16384, px=5.0, nodata=0.0, dtype="uint8", tile=4096, f32_too=True),
        # the same product on a ragged raster with NoData (the common real DEM)
        dict(name="job_topousm_nodata", kind="job", algo="topousm_fast", mode="spatial", h=9001,
             w=7003, px=10.0, nodata=0.01, dtype="float32", tile=4096),
        # openness with its default 16 directions and p1/p99 stretch pre-pass
        dict(name="job_openness", kind="job", algo="openness", mode="local", h=8192, w=6144,
             px=10.0, nodata=0.0, dtype="float32", tile=4096),
        # the default (spatial) mode of a stencil: Gaussian, decimated and overview radii
        dict(name="job_hillshade_spatial", kind="job", algo="hillshade", mode="spatial", h=8192,
             w=8192, px=5.0, nodata=0.0, dtype="float32", tile=4096),
        # the default mode of ambient occlusion, quantised output
        dict(name="job_ao_spatial", kind="job", algo="ambient_occlusion", mode="spatial", h=5003,
             w=6007, px=10.0, nodata=0.0, dtype="uint8", tile=4096),
        # the largest: curvature + openness of one raster with NoData, captured and replayed
        dict(name="raster_job_curv_open", kind="raster_job", h=20011, w=16001, px=10.0,
             nodata=0.01, tile=4096),
        # ragged projected and geographic tiles, four products each, one batch
        dict(name="batch_ragged_tiles", kind="batch", n=64, lo=256, hi=3000),
        # surrogate inference at the radius it was trained for
        dict(name="surrogate_8192", kind="surrogate", h=8192, w=8192, px=10.0),
        # one training step's forward and backward passes
        dict(name="surrogate_train_step", kind="train", batch=32, side=80),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["tile", "tile", "tile", "job", "job", "job", "job", "batch",
                       "raster_job", "surrogate", "train"])
    px = rng.choice([2.0, 5.0, 10.0, 30.0])
    nodata = rng.choice([0.0, 0.01])
    if kind == "tile":
        c = dict(kind=kind, algo=rng.choice(["hillshade", "slope", "curvature", "topousm_fast",
                                             "openness", "ambient_occlusion"]),
                 h=_log_uniform(rng, 128, 4096), w=_log_uniform(rng, 128, 4096), px=px,
                 nodata=nodata)
    elif kind == "job":
        algo = rng.choice(["hillshade", "slope", "curvature", "topousm_fast", "openness",
                           "ambient_occlusion"])
        mode = "spatial" if algo == "topousm_fast" else rng.choice(["local", "spatial"])
        hi = 6000 if mode == "spatial" else 10000
        c = dict(kind=kind, algo=algo, mode=mode, h=_log_uniform(rng, 1100, hi),
                 w=_log_uniform(rng, 1100, hi), px=px, nodata=nodata,
                 dtype=rng.choice(["float32", "int16", "uint8"]),
                 tile=rng.choice([2048, 4096]))
    elif kind == "raster_job":
        return dict(kind=kind, h=_log_uniform(rng, 2100, 12000), w=_log_uniform(rng, 2100, 12000),
                    px=px, nodata=nodata, tile=rng.choice([2048, 4096]))
    elif kind == "batch":
        return dict(kind=kind, n=rng.randint(8, 64), lo=rng.choice([128, 256, 300]),
                    hi=rng.randint(800, 3000))
    elif kind == "surrogate":
        return dict(kind=kind, h=16 * _log_uniform(rng, 140, 512),
                    w=16 * _log_uniform(rng, 140, 512), px=px)
    else:
        return dict(kind=kind, batch=rng.randint(4, 32), side=rng.randint(48, 80))
    if c["algo"] == "curvature":
        # planform and profile divide by a vanishing gradient: no tolerance holds there
        c["curvature_type"] = rng.choice(["mean", "gaussian"])
    if c["algo"] == "openness":
        c["openness_type"] = rng.choice(["positive", "negative"])
    return c


# --------------------------------------------------------------- inputs and run

def _terrain(h, w, seed, hurst=0.75, relief=2500.0):
    """fBm of the next power of two, cropped (the FFT library meets few sizes)."""
    big = 1 << max(8, (max(h, w) - 1).bit_length())
    return synth.fbm(big, big, hurst, relief, seed=seed, device="cuda")[:h, :w].contiguous()


def _raster(case, seed, sentinel):
    dem = _terrain(case["h"], case["w"], seed)
    if case.get("nodata"):
        synth.apply_discs(dem, synth.nodata_discs(case["h"], case["w"], case["nodata"], seed + 1),
                          sentinel)
    return dem


def _tile_params(case):
    p = {"pixel_size": case["px"]}
    if case["algo"] == "curvature":
        p["curvature_type"] = case.get("curvature_type", "mean")
    if case["algo"] == "openness":
        p["openness_type"] = case.get("openness_type", "positive")
        p["global_stats"] = (0.55, 0.4)
    if case["algo"] == "ambient_occlusion":
        p["global_stats"] = (0.45, 0.5)
    if case["algo"] == "topousm_fast":
        p["global_stats"] = (USM_SCALE,)
    return p


_BATCH_RADII = [2, 8, 32, 128]
_BATCH_WEIGHTS = [8 / 15, 4 / 15, 2 / 15, 1 / 15]


def _metres_per_degree(lat):
    """WGS84 series: metres per degree of longitude and latitude."""
    a = np.radians(lat)
    return (111412.84 * np.cos(a) - 93.5 * np.cos(3 * a) + 0.118 * np.cos(5 * a),
            111132.92 - 559.82 * np.cos(2 * a) + 1.175 * np.cos(4 * a) - 0.0023 * np.cos(6 * a))


def _batch_geometry(case):
    """Per tile: side, Hurst exponent, relief, and for odd (geographic) tiles the
    x cell width of every row and the y cell size of 1 arc-second cells."""
    out = []
    for i in range(case["n"]):
        r = np.random.default_rng([case["n"], case["lo"], case["hi"], i])
        side = int(round(math.exp(r.uniform(math.log(case["lo"]), math.log(case["hi"])))))
        hurst, relief = float(r.uniform(0.6, 0.9)), float(r.uniform(500.0, 3000.0))
        rows = sy = None
        if i % 2:
            lat = float(r.uniform(30.0, 60.0))
            rows = _metres_per_degree(lat + (0.5 * side - 0.5 - np.arange(side)) / 3600.0)[0]
            rows, sy = rows / 3600.0, float(_metres_per_degree(lat)[1]) / 3600.0
        out.append((side, hurst, relief, rows, sy))
    return out


def _batch_tiles(case, seed):
    return [(_terrain(side, side, seed + 7 * i, hurst, relief), rows, sy)
            for i, (side, hurst, relief, rows, sy) in enumerate(_batch_geometry(case))]


def _train_inputs(case, seed):
    """A batch of pyramid features (bf16 bits, four of eight channels in use) and
    the loss gradient at the two output channels of the labelled centre."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    b, n = case["batch"], case["side"]
    x = torch.zeros((b, n, n, 8), device="cuda")
    x[..., :4] = torch.randn((b, n, n, 4), generator=g, device="cuda") * 0.5
    dz = torch.zeros((b, n, n, 32), device="cuda")
    dz[:, 8:-8, 8:-8, :2] = torch.randn((b, n - 16, n - 16, 2), generator=g, device="cuda") * 1e-3
    return (x.to(torch.bfloat16).view(torch.int16), dz.to(torch.bfloat16).view(torch.int16))


def prepare(case, seed):
    k = case["kind"]
    if k == "tile":
        return dict(k=k, algo=ALGORITHMS[case["algo"]], dem=_raster(case, seed, float("nan")),
                    params=_tile_params(case))
    if k == "job":
        dem = _raster(case, seed, NODATA)
        kw = dict(mode=case["mode"], tile_size=case["tile"], pixel_size=case["px"],
                  output_dtype=case["dtype"], nodata=NODATA if case["nodata"] else None)
        for key in ("curvature_type", "openness_type"):
            if key in case:
                kw[key] = case[key]
        if case.get("f32_too"):
            # the headline call: both encodings into the caller's rasters
            kw.update(out=torch.empty(dem.shape, dtype=torch.uint8, device="cuda"),
                      out_f32=torch.empty_like(dem), copy_input=False)
        return dict(k=k, algo=case["algo"], dem=dem, kw=kw)
    if k == "raster_job":
        dem = _raster(case, seed, NODATA)
        job = RasterJob(dem, {"curvature": {"curvature_type": "mean", "mode": "local"},
                              "openness": {"openness_type": "positive", "num_directions": 8,
                                           "max_distance": 64, "mode": "local"}},
                        tile_size=case["tile"], pixel_size=case["px"],
                        nodata=NODATA if case["nodata"] else None)
        job.set_split(True)           # the shape the job's own tuner picks
        job.capture()
        return dict(k=k, job=job)
    if k == "batch":
        jobs, at = [], 0
        tiles = _batch_tiles(case, seed)
        # one buffer per product for the whole batch, each tile a view of it
        pools = torch.empty((4, sum(t[0].numel() for t in tiles)), device="cuda")
        for dem, rows, sy in tiles:
            p = {"radii": list(_BATCH_RADII), "weights": list(_BATCH_WEIGHTS),
                 "curvature_type": "mean", "global_stats": (USM_SCALE,), "pixel_size": 10.0}
            if rows is not None:
                p.update(pixel_scale_x_rows=rows, pixel_scale_y=-sy,
                         pixel_size=0.5 * (float(rows.mean()) + sy))
            hs, sl, cv, usm = (q[at:at + dem.numel()].view(dem.shape) for q in pools)
            at += dem.numel()
            jobs.append(TileJob(dem=dem, params=p, hillshade=hs, slope=sl, curvature=cv,
                                topousm=usm, nan_free=True))
        return dict(k=k, pools=pools, batch=FusedBatch(jobs))
    if k == "surrogate":
        net = Net("cuda")
        net.load(WEIGHTS_FILE)
        return dict(k=k, net=net, px=case["px"], dem=_terrain(case["h"], case["w"], seed))
    net = Net("cuda")
    net.load(WEIGHTS_FILE)
    x, dz = _train_inputs(case, seed)
    return dict(k=k, net=net, x=x, dz=dz)


def run(s):
    if s["k"] == "tile":
        return s["algo"].process(s["dem"], **s["params"])
    if s["k"] == "job":
        out, _ = process_dem(s["dem"], s["algo"], **s["kw"])
        return (out, s["kw"]["out_f32"]) if "out_f32" in s["kw"] else out
    if s["k"] == "raster_job":
        s["job"].replay()
        return dict(s["job"].outputs)
    if s["k"] == "batch":
        s["batch"].run()
        return tuple(s["pools"])
    if s["k"] == "surrogate":
        return surrogate_openness(s["net"], s["dem"], 1024, 16, s["px"])
    yf, acts, pres = s["net"].forward(s["x"], keep=True)
    s["net"].backward(acts, pres, s["dz"])
    return yf, s["net"].grad


# ------------------------------------------------------------------------- work

_OUT_BYTES = {"float32": 4, "int16": 2, "uint8": 1}
# float operations of one output pixel that the formula itself has
_PIXEL_FLOPS = {"hillshade": 16, "slope": 10, "curvature": 45, "topousm_fast": 60,
                "openness": 16 * 10 * 3, "ambient_occlusion": 64 * 5}


def work(case):
    k = case["kind"]
    if k == "train":
        cells = case["batch"] * case["side"] ** 2
        macs = 9 * (4 * 32 + 4 * 32 * 32 + 32 * 2)      # a forward pass per cell
        return {"bytes": cells * (4 * 2 + 2 * 2 + 2 * 4) + 2 * 4 * macs,
                "flops": cells * 2 * 3 * macs}
    if k == "batch":
        n = sum(g[0] ** 2 for g in _batch_geometry(case))
        return {"bytes": 20 * n, "flops": n * (16 + 10 + 45 + 60)}
    n = case["h"] * case["w"]
    if k == "surrogate":
        macs = 9 * (4 * 32 + 4 * 32 * 32 + 32 * 2)
        return {"bytes": 8 * n, "flops": n // 64 * 2 * macs + n * 12}
    if k == "raster_job":
        return {"bytes": 12 * n, "flops": n * (45 + 8 * 10 * 3)}
    out = _OUT_BYTES[case.get("dtype", "float32")] + (4 if case.get("f32_too") else 0)
    flops = _PIXEL_FLOPS[case["algo"]]
    if case.get("mode") == "spatial" and case["algo"] != "topousm_fast":
        radii = _auto_radii(min(case["h"], case["w"]))
        flops *= len(radii)
        if case["algo"] in _STENCILS:
            # two symmetric filter passes of 2 r taps a side at full resolution
            flops += sum(12 * r for r in radii if r < 48)
    return {"bytes": n * (4 + out), "flops": n * flops}


# -------------------------------------------------------------------- tolerance

def tolerance(case):
    """About four times the largest distance from the float64 results seen over the listed
    and about 130 drawn cases.  Differences of float32 heights set the stencils' figures
    (curvature's most), float32 means TopoUSM's and the smoothed radii's, and bf16
    activations the network's.  Quantised rasters round near ties either way; the finer
    int16 step meets more of them, most of all where the p1/p99 stretch or the
    smoothed heights differ in their last bits."""
    k = case["kind"]
    if k != "tile" and k != "job":
        return {"rel": {"batch": 9e-5, "raster_job": 1.6e-4, "surrogate": 9e-5,
                        "train": 2e-2}[k]}
    spatial = case.get("mode") == "spatial"
    dtype = case.get("dtype", "float32")
    if dtype == "int16":
        return {"rel": 3e-4, "differ": 0.35} if spatial else {"rel": 3e-5, "differ": 0.03}
    if dtype == "uint8":
        return {"rel": 8e-4, "differ": 2e-3} if spatial else {"rel": 3e-4, "differ": 5e-4}
    if spatial:
        return {"rel": 3e-5}
    return {"rel": {"hillshade": 5e-6, "slope": 5e-6, "curvature": 3e-5, "topousm_fast": 1.5e-5,
                    "openness": 4e-6, "ambient_occlusion": 4e-6}[case["algo"]]}


# ------------------------------------------------- float64 results in plain torch
#
# Windows are float64 tensors with NaN for NoData.  The rules (edges, NaN-aware
# means, decimation, tile geometry) are the framework's; the arithmetic is 64-bit.

_STENCILS = ("hillshade", "slope", "curvature")
_RAYS = ("openness", "ambient_occlusion")
_GAMMA = 1 / 2.2


def _edge_index(n, lo, hi, mode, dev):
    i = torch.arange(lo, hi, device=dev)
    if mode == "nearest":
        return i.clamp(0, n - 1)
    i = i % (2 * n)                                  # symmetric: d c b a | a b c d | d c b a
    return torch.where(i < n, i, 2 * n - 1 - i)


def _pad(x, p, mode):
    r = _edge_index(x.shape[0], -p, x.shape[0] + p, mode, x.device)
    c = _edge_index(x.shape[1], -p, x.shape[1] + p, mode, x.device)
    return x[r][:, c]


def _gauss(x, sigma):
    rad = int(4.0 * sigma + 0.5)
    g = np.exp(-0.5 / (sigma * sigma) * np.arange(rad + 1, dtype=np.float64) ** 2)
    g = g / (g[0] + 2 * g[1:].sum())
    for _ in range(2):                               # axis 0, then axis 1 by transposing
        h = x.shape[0]
        y = x[_edge_index(h, -rad, h + rad, "nearest", x.device)]
        acc = y[rad:rad + h] * float(g[0])
        for d in range(1, rad + 1):
            acc += (y[rad - d:rad - d + h] + y[rad + d:rad + d + h]) * float(g[d])
        x = acc.T
    return x


def _box(x, r):
    n = 2 * r + 1
    for _ in range(2):
        h = x.shape[0]
        c = torch.cumsum(x[_edge_index(h, -r, h + r, "reflect", x.device)], 0)
        m = c[n - 1:].clone()
        m[1:] -= c[:-n]
        x = (m / n).T
    return x


def _nan_mean(x, f):
    bad = torch.isnan(x)
    if not bool(bad.any()):
        return f(x)
    sv, sw = f(torch.where(bad, 0.0, x)), f((~bad).to(x.dtype))
    return torch.where(sw > 1e-12, sv / sw.clamp_min(1e-300), torch.zeros_like(sv))


def _diff0(f, step):
    """d/drow, second order at both ends."""
    d = torch.empty_like(f)
    d[1:-1] = (f[2:] - f[:-2]) / 2
    d[0] = -1.5 * f[0] + 2 * f[1] - 0.5 * f[2]
    d[-1] = 1.5 * f[-1] - 2 * f[-2] + 0.5 * f[-3]
    return d / step


def _gradient(f, sy, sx):
    dx = _diff0(f.T, 1.0).T
    return _diff0(f, sy), dx / (sx[:, None] if isinstance(sx, torch.Tensor) else sx)


def _scales(p):
    """Signed x and y cell sizes; x may be a per-row tensor."""
    px = p["pixel_size"]
    sx = p.get("sx", px)
    if isinstance(sx, np.ndarray):
        sx = torch.from_numpy(sx).cuda()
    return sx, p.get("sy", px)


def _filled_gradient(x, p):
    bad = torch.isnan(x)
    if bool(bad.any()):
        x = torch.where(bad, _nan_mean(x, lambda a: _gauss(a, 1.0)), x)
    sx, sy = _scales(p)
    return _gradient(x, abs(sy), abs(sx)) + (bad,)


def _hillshade(x, p):
    dy, dx, bad = _filled_gradient(x, p)
    sx, sy = _scales(p)
    sx = float(sx[0]) if isinstance(sx, torch.Tensor) else sx
    e, n = dx * math.copysign(1, sx), dy * math.copysign(1, sy)
    az, al = math.radians(315.0), math.radians(45.0)
    hs = (-e * (math.sin(az) * math.cos(al)) - n * (math.cos(az) * math.cos(al)) + math.sin(al))
    hs = (hs / torch.sqrt(e * e + n * n + 1)).clamp(0, 1)
    return hs.masked_fill(bad, float("nan"))


def _slope(x, p):
    dy, dx, bad = _filled_gradient(x, p)
    return torch.rad2deg(torch.atan(torch.hypot(dx, dy))).masked_fill(bad, float("nan"))


def _curvature(x, p):
    q, pp, bad = _filled_gradient(x, p)
    sx, sy = _scales(p)
    dyy, dyx = _gradient(q, sy, sx)
    dxy, dxx = _gradient(pp, sy, sx)
    g = 1 + pp * pp + q * q
    if p.get("curvature_type", "mean") == "mean":
        num = (1 + q * q) * dxx - pp * q * (dxy + dyx) + (1 + pp * pp) * dyy
        c = -num / (2 * g ** 1.5 + 1e-10)
    else:
        c = (dxx * dyy - dxy * dxy) / (g * g)
    return (((torch.tanh(100 * c) + 1) / 2) ** _GAMMA).masked_fill(bad, float("nan"))


def _factor(r, px, algo):
    k = {"topousm_fast": 1.15, "curvature": 1.1, "ambient_occlusion": 1.5,
         "openness": 1.4}.get(algo, 1.0)
    score = max(1.0, float(r)) / 24.0 * k * max(1.0, 1.0 / max(1e-3, px)) ** 0.35
    return 1 if score <= 1 else int(min(16, 2 ** int(math.floor(math.log2(score)))))


def _decimate(x, f):
    if f <= 1:
        return x
    h, w = x.shape
    oh, ow = -(-h // f), -(-w // f)
    y = torch.full((oh * f, ow * f), float("nan"), dtype=x.dtype, device=x.device)
    y[:h, :w] = x
    y = y.view(oh, f, ow, f)
    ok = torch.isfinite(y)
    n = ok.sum(dim=(1, 3))
    s = torch.where(ok, y, 0.0).sum(dim=(1, 3)) / n.clamp_min(1)
    s = torch.where(n > 0, s, float("nan"))
    bad = torch.isnan(s)
    if bool(bad.any()):                              # voids enclosed by data are filled
        sig = max(1.0, min(oh, ow) / 64.0)
        sv = _gauss(torch.where(bad, 0.0, s), sig)
        sw = _gauss((~bad).to(s.dtype), sig)
        s = torch.where(bad & (sw > 0.5), sv / sw.clamp_min(1e-6), s)
    return s


def _lerp_axis0(x, pos):
    i = pos.floor().long().clamp(0, x.shape[0] - 1)
    j = (i + 1).clamp(max=x.shape[0] - 1)
    t = (pos - i)[:, None]
    return x[i] * (1 - t) + x[j] * t


def _corner_zoom(x, h, w):
    """Order-1 zoom with aligned corners, NaN cells carrying no weight."""
    if tuple(x.shape) == (h, w):
        return x

    def z(a):
        for n, o in ((a.shape[0], h), (a.shape[1], w)):
            pos = torch.arange(o, device=a.device, dtype=torch.float64)
            a = _lerp_axis0(a, pos * ((n - 1) / (o - 1) if o > 1 else 0.0)).T
        return a
    bad = torch.isnan(x)
    if not bool(bad.any()):
        return z(x)
    num, den = z(torch.where(bad, 0.0, x)), z((~bad).to(x.dtype))
    return torch.where(den > 1e-3, num / den.clamp_min(1e-6), float("nan"))


def _centre_sample(x, r0, r1, c0, c1, fh, fw):
    """Bilinear sample of an overview at raster pixels.  The positions are float32
    values by definition, as the rule that the overview users follow has them."""
    for lo, hi, n, full in ((r0, r1, x.shape[0], fh), (c0, c1, x.shape[1], fw)):
        pos = ((torch.arange(lo, hi, device=x.device, dtype=torch.float32) + 0.5)
               * float(np.float32(n / float(full))) - 0.5)
        x = _lerp_axis0(x, pos.double().clamp(0, n - 1)).T
    return x


def _area_matrix(n, m):
    """m x n overlap weights of n cells with m equal intervals."""
    edge = torch.arange(m + 1, device="cuda", dtype=torch.float64) * (n / m)
    c = torch.arange(n, device="cuda", dtype=torch.float64)
    return (torch.minimum(edge[1:, None], c + 1) - torch.maximum(edge[:-1, None], c)).clamp_min(0)


def _overview(x):
    h, w = x.shape
    scale = max(w / 2048, h / 2048, 1.0)
    oh, ow = int(round(h / scale)), int(round(w / scale))
    if (oh, ow) == (h, w):
        return x, scale
    ok = torch.isfinite(x)
    a, b = _area_matrix(h, oh), _area_matrix(w, ow).T
    num = (a @ torch.where(ok, x, 0.0)) @ b
    den = (a @ ok.to(x.dtype)) @ b
    return torch.where(den > 1e-9, num / den.clamp_min(1e-300), float("nan")), scale


def _topousm(x, radii, weights, px):
    """sum of w_i (z - mean_i), NaN kept."""
    acc = torch.zeros_like(x)
    for r, wt in zip(radii, weights):
        f = _factor(r, px, "topousm_fast")
        y = _decimate(x, f)
        rc = max(1, int(round(r / f))) if f > 1 else int(r)
        m = _nan_mean(y, (lambda a: _gauss(a, 1.0)) if rc <= 1 else (lambda a: _box(a, rc)))
        acc += wt * (x - _corner_zoom(m, *x.shape))
    return acc


def _steps(p):
    sx, sy = _scales(p)
    return abs(sx), abs(sy)


def _openness(x, p):
    h, w = x.shape
    n, dist = p.get("num_directions", 16), p.get("max_distance", 50)
    rs = np.unique((np.linspace(0.1, 1.0, 10) * dist).astype(int))
    rs = rs[rs > 0]
    d = int(rs.max())
    sx, sy = _steps(p)
    neg = p.get("openness_type", "positive") == "negative"
    y = torch.full((h + 2 * d, w + 2 * d), float("nan"), dtype=x.dtype, device=x.device)
    y[d:d + h, d:d + w] = x
    total, count = torch.zeros_like(x), torch.zeros_like(x)
    for ang in np.linspace(0, 2 * np.pi, int(n), endpoint=False):
        ext = torch.full_like(x, float("nan"))
        for r in rs:
            ox, oy = int(round(float(r) * np.cos(ang))), int(round(float(r) * np.sin(ang)))
            if ox == 0 and oy == 0:
                continue
            q = (y[d + oy:d + oy + h, d + ox:d + ox + w] - x) / math.hypot(ox * sx, oy * sy)
            ext = torch.fmin(ext, q) if neg else torch.fmax(ext, q)
        ok = ~torch.isnan(ext)
        a = torch.atan(ext)
        total += torch.where(ok, math.pi / 2 + (a if neg else -a), 0.0)
        count += ok
    total /= count.clamp_min(1)
    if p.get("degrees"):
        return torch.rad2deg(total).masked_fill(torch.isnan(x), float("nan"))
    v = (total / (math.pi / 2)).clamp(0, 1) ** _GAMMA
    return v.masked_fill(torch.isnan(x), float("nan"))


def _ao(x, p):
    h, w = x.shape
    radius = float(p.get("radius", 10.0))
    d = max(1, int(round(radius)))
    y = _pad(x, d, "nearest")
    sx, sy = _steps(p)
    ang = np.linspace(0, 2 * np.pi, int(p.get("num_samples", 16)), endpoint=False)
    total, count = torch.zeros_like(x), torch.zeros_like(x)
    for rf in (0.25, 0.5, 0.75, 1.0):
        for ox, oy in zip(np.round(radius * rf * np.cos(ang)).astype(int),
                          np.round(radius * rf * np.sin(ang)).astype(int)):
            if ox == 0 and oy == 0:
                continue
            v = y[d + oy:d + oy + h, d + ox:d + ox + w]
            a = torch.atan((v - x) / math.hypot(ox * sx, oy * sy)).clamp(0, math.pi / 4)
            ok = ~torch.isnan(a)
            total += torch.where(ok, a * ((1 - 0.3 * rf) / (math.pi / 4)), 0.0)
            count += ok
    v = (1 - total / count.clamp_min(1)).clamp(0, 1)
    bad = torch.isnan(x)
    return (_gauss(torch.where(bad, 1.0, v), 1.0) ** _GAMMA).masked_fill(bad, float("nan"))


_LOCAL = {"hillshade": _hillshade, "slope": _slope, "curvature": _curvature,
          "openness": _openness, "ambient_occlusion": _ao}


def _scaled(p, f):
    q = dict(p, pixel_size=p["pixel_size"] * f)
    for k in ("sx", "sy"):
        if k in q:
            q[k] = q[k] * f
    return q


def _spatial_block(algo, x, r, p):
    """The local function at one radius: of the smoothed block for the stencils, of
    the block (decimated for the larger radii) for the ray algorithms."""
    f = _factor(r, p["pixel_size"], algo)
    if algo in _STENCILS:
        if r > 1:
            y = _decimate(x, f)
            y = _nan_mean(y, lambda a: _gauss(a, max(0.5, r / f / 2)))
            x = _corner_zoom(y, *x.shape)
        return _LOCAL[algo](x, p)
    y, q, rr = x, p, r
    if f > 1:
        y, q = _decimate(x, f), _scaled(p, f)
        rr = max(2, int(round(r / f))) if algo == "openness" else max(1.0, r / f)
    key = "max_distance" if algo == "openness" else "radius"
    return _corner_zoom(_LOCAL[algo](y, dict(q, **{key: rr})), *x.shape)


def _spatial_tile(algo, x, p, radii, weights, ov, origin, full):
    h, w = x.shape
    acc = None
    for r, wt in zip(radii, weights):
        if r > max(256, min(h, w) // 16):
            dec = 0.5 * (full[1] / ov.shape[1] + full[0] / ov.shape[0])
            key = (r, dec)
            cache = p["cache"]
            if key not in cache:
                cache[key] = _spatial_block(algo, ov, max(1, int(round(r / dec))),
                                            _scaled(p, dec))
            f = _centre_sample(cache[key], origin[0], origin[0] + h, origin[1], origin[1] + w,
                               *full)
            f = f.masked_fill(torch.isnan(x), float("nan"))
        else:
            d = int(r) + 1 if algo in _RAYS else (
                max(3, 2 * r + 2) if algo == "curvature" else max(2, 2 * r + 1))
            d = max(1, min(d, min(h, w) - 1))
            f = _spatial_block(algo, _pad(x, d, "reflect"), r, p)[d:d + h, d:d + w]
        acc = f * wt if acc is None else acc + f * wt
    return acc


def _auto_radii(short):
    return [r for r in (2, 8, 32, 128, 512, 2048) if r <= min(2048.0, short / 10.0)] or [2]


def _halving(n):
    raw = [2.0 ** (n - 1 - i) for i in range(n)]
    return [v / sum(raw) for v in raw]


def _tiles(h, w, tile, pad):
    for cy in range(0, h, tile):
        for cx in range(0, w, tile):
            ch, cw = min(tile, h - cy), min(tile, w - cx)
            wy, wx = max(cy - pad, 0), max(cx - pad, 0)
            yield (cy, cx, ch, cw, wy, wx, min(cy + ch + pad, h) - wy,
                   min(cx + cw + pad, w) - wx)


def _percentile(v, q):
    v = torch.sort(v).values
    pos = q / 100.0 * (v.numel() - 1)
    i = int(math.floor(pos))
    a, b = float(v[i]), float(v[min(i + 1, v.numel() - 1)])
    return a + (b - a) * (pos - i)


def _prepass_values(dem, scale_px, block):
    """The pooled values of the 3 x 3 stratified statistics windows."""
    h, w = dem.shape
    cov = max(1, max(h, w) // 512)
    oh, ow = max(1, h // cov), max(1, w // cov)
    ri = torch.from_numpy(np.minimum(np.floor((np.arange(oh) + 0.5) * (h / oh)), h - 1)).long()
    ci = torch.from_numpy(np.minimum(np.floor((np.arange(ow) + 0.5) * (w / ow)), w - 1)).long()
    ok = torch.isfinite(dem[ri.cuda()][:, ci.cuda()]).cpu().numpy()
    ys, xs = np.nonzero(ok.any(1))[0], np.nonzero(ok.any(0))[0]
    y0, y1 = int(ys[0]) * cov, min(h, (int(ys[-1]) + 1) * cov)
    x0, x1 = int(xs[0]) * cov, min(w, (int(xs[-1]) + 1) * cov)
    margin = int(scale_px + 16)
    t = min(max(2048, 4 * margin), max(h, w))
    gh, gw = max(1, (y1 - y0) // 3), max(1, (x1 - x0) // 3)
    seen, pool = [], []
    for gy in range(3):
        for gx in range(3):
            wy = min(max(0, y0 + gy * gh + gh // 2 - t // 2), max(0, h - t))
            wx = min(max(0, x0 + gx * gw + gw // 2 - t // 2), max(0, w - t))
            th, tw = min(t, h - wy), min(t, w - wx)
            if (wy, wx, th, tw) in seen:
                continue
            seen.append((wy, wx, th, tw))
            m = min(margin, th // 3, tw // 3)
            v = block(dem[wy:wy + th, wx:wx + tw].double())[m:th - m, m:tw - m].reshape(-1)
            pool.append(v[torch.isfinite(v)])
    return torch.cat(pool)


_RANGE = {"hillshade": (0.0, 1.0), "slope": (0.0, 90.0), "curvature": (0.0, 1.0),
          "openness": (0.0, 1.0), "ambient_occlusion": (0.0, 1.0),
          "topousm_fast": (-1.176, 1.176)}


def _quantised(v, algo, dtype):
    lo, hi = _RANGE[algo]
    top = {"int16": 32767, "uint8": 255}[dtype]
    if lo < 0:
        a, b, lo_dn = ((top / hi, 0.0, -top) if dtype == "int16"
                       else ((top - 1) / 2.0 / hi, (top + 1) / 2.0, 1))
    else:
        a = (top - 1) / (hi - lo)
        b, lo_dn = 1.0 - a * lo, 1
    q = torch.round(v * a + b).clamp(lo_dn, top)
    return torch.where(torch.isnan(v), 0.0, q).to(getattr(torch, dtype))


def _exact_job(dem, algo, mode, px, tile, opts):
    """The float64 raster of one scheduler job, before any quantisation."""
    h, w = dem.shape
    p = dict(opts, pixel_size=px, sx=px, sy=-px, cache={})
    radii = _auto_radii(min(h, w)) if mode == "spatial" else [1]
    weights = _halving(len(radii))
    switch = max(256, tile // 16)
    pad, ov, field, stats = 64, None, None, None
    small = [(r, v) for r, v in zip(radii, weights) if r <= switch]
    large = [(r, v) for r, v in zip(radii, weights) if r > switch]
    if algo == "topousm_fast":
        stats = _percentile(_prepass_values(
            dem, max(radii), lambda x: _topousm(x, radii, weights, px)).abs(), 99.0)
        pad = max(64, -(-(max(r for r, _ in small) + 16) // 32) * 32)
        if large:
            ov, scale = _overview(dem.double())
            field = 0
            for r, v in large:
                rc = max(1, int(round(r / scale)))
                field = field + v * _nan_mean(
                    ov, (lambda a: _gauss(a, 1.0)) if rc <= 1 else (lambda a: _box(a, rc)))
    elif algo in _RAYS:
        top = max(max(radii), p.get("max_distance", 50) if algo == "openness" else 10.0)
        v = _prepass_values(dem, top, lambda x: _LOCAL[algo](x, p))
        lo, hi = _percentile(v, 1.0), _percentile(v, 99.0)
        stats = (lo, hi - lo)
    if mode == "spatial" and algo != "topousm_fast":
        rm = max(r for r, _ in small)
        need = rm + 16 if algo in _RAYS else 2 * rm + 2
        pad = max(64, -(-need // 32) * 32)
        ov, _ = _overview(dem.double())
    out = torch.empty((h, w), dtype=torch.float64, device=dem.device)
    for cy, cx, ch, cw, wy, wx, wh, ww in _tiles(h, w, tile, pad):
        x = dem[wy:wy + wh, wx:wx + ww].double()
        if algo == "topousm_fast":
            v = _topousm(x, [r for r, _ in small], [s for _, s in small], px)
            if large:
                v = v + sum(s for _, s in large) * x - _centre_sample(
                    field, wy, wy + wh, wx, wx + ww, h, w)
            v = v / stats
        elif mode == "spatial":
            v = _spatial_tile(algo, x, p, radii, weights, ov, (wy, wx), (h, w))
        else:
            v = _LOCAL[algo](x, p)
        out[cy:cy + ch, cx:cx + cw] = v[cy - wy:cy - wy + ch, cx - wx:cx - wx + cw]
    if algo in _RAYS and stats[1] > 1e-12:
        out = ((out - stats[0]) / stats[1]).clamp_min(0)
    return out


def _conv(x, w, b):
    """3 x 3 correlation with zero padding, channels last."""
    n, h, wd, _ = x.shape
    y = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
    out = torch.zeros((n, h, wd, w.shape[0]), dtype=x.dtype, device=x.device)
    for i in range(3):
        for j in range(3):
            out = out + y[:, i:i + h, j:j + wd] @ w[:, :, i, j].T
    return out + b


def _network(x, flat):
    widths, o, layers = (8, 32, 32, 32, 32, 32, 2), 0, []
    for ci, co in zip(widths[:-1], widths[1:]):
        w = flat[o:o + co * ci * 9].view(co, ci, 3, 3)
        layers.append((w, flat[o + co * ci * 9:o + co * ci * 9 + 32][:co]))
        o += co * ci * 9 + 32
    for i, (w, b) in enumerate(layers):
        x = _conv(x, w, b)
        if i < 5:
            x = x * torch.sigmoid(2 * math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3))
    return x


def _weights64():
    with np.load(os.path.join(os.path.dirname(synth.__file__), "data",
                              "openness_surrogate_r1024.npz"), allow_pickle=False) as z:
        return torch.from_numpy(z["flat"].astype(np.float64)).cuda()


def _centre_zoom(x, f):
    for _ in range(2):
        n = x.shape[0]
        pos = ((torch.arange(n * f, device=x.device, dtype=torch.float64) + 0.5) / f - 0.5)
        x = _lerp_axis0(x, pos.clamp(0, n - 1)).T
    return x


def _exact_surrogate(dem, px):
    z = dem.double()
    zg = z.view(z.shape[0] // 8, 8, z.shape[1] // 8, 8).mean(dim=(1, 3))
    z16 = zg.view(zg.shape[0] // 2, 2, zg.shape[1] // 2, 2).mean(dim=(1, 3))
    base = _centre_zoom(_openness(z16, {"pixel_size": px * 16, "max_distance": 64,
                                        "num_directions": 16, "degrees": True}), 2)
    x = torch.zeros((1,) + tuple(zg.shape) + (8,), dtype=torch.float64, device="cuda")
    for k, r in enumerate((16, 64, 256, 1024)):
        x[0, ..., k] = (_box(zg, r // 8) - zg) * (10.0 / (r * px))
    y = _network(x, _weights64())[0]
    s = torch.repeat_interleave(torch.repeat_interleave(y[..., 1], 8, 0), 8, 1)
    return _centre_zoom(y[..., 0] + base, 8) + s / 20.0 * (z - _centre_zoom(zg, 8))


def exact(case, seed):
    k = case["kind"]
    if k == "train":
        x, dz = (t.view(torch.bfloat16).double() for t in _train_inputs(case, seed))
        flat = _weights64().requires_grad_(True)
        y = _network(x, flat)
        y.backward(dz[..., :2])
        return y.detach(), flat.grad
    if k == "surrogate":
        return _exact_surrogate(_terrain(case["h"], case["w"], seed), case["px"])
    if k == "batch":
        out = []
        for dem, rows, sy in _batch_tiles(case, seed):
            p = {"pixel_size": 10.0}
            if rows is not None:
                p = {"pixel_size": 0.5 * (float(rows.mean()) + sy), "sx": rows, "sy": -sy}
            x = dem.double()
            out.append((_hillshade(x, p), _slope(x, p), _curvature(x, p),
                        _topousm(x, _BATCH_RADII, _BATCH_WEIGHTS, p["pixel_size"]) / USM_SCALE))
        return tuple(torch.cat([v[i].reshape(-1) for v in out]) for i in range(4))
    dem = _raster(case, seed, float("nan"))
    if k == "raster_job":
        return {"curvature": _exact_job(dem, "curvature", "local", case["px"], case["tile"], {}),
                "openness": _exact_job(dem, "openness", "local", case["px"], case["tile"],
                                       {"num_directions": 8, "max_distance": 64})}
    opts = {key: case[key] for key in ("curvature_type", "openness_type") if key in case}
    if k == "job":
        v = _exact_job(dem, case["algo"], case["mode"], case["px"], case["tile"], opts)
        if case["dtype"] == "float32":
            return v
        q = _quantised(v, case["algo"], case["dtype"])
        return (q, v) if case.get("f32_too") else q
    p = _tile_params(case)
    x = dem.double()
    if case["algo"] == "topousm_fast":
        radii = sorted({max(2, min(int(d / case["px"]), 256)) for d in (5, 20, 80, 320)})
        return _topousm(x, radii, [1.0 / len(radii)] * len(radii), case["px"]) / USM_SCALE
    v = _LOCAL[case["algo"]](x, p)
    if "global_stats" in p:
        v = ((v - p["global_stats"][0]) / p["global_stats"][1]).clamp_min(0)
    return v
