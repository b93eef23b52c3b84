"""The work that a user of this framework has it do, as cases that can be timed.

``listed()`` names the cases, ``draw(rng)`` gives one more of the same ranges, ``prepare`` makes what a
program holds before the call (the chunk, the CF tables, the plan), ``run`` is one pass through the public
entry points and ``exact`` is what that pass computes, in 64 bits and plain torch.

The calls (``do``):
  put, get     the drop-in functions on numpy arrays, one facet of one chunk, as ClassDDEGridMachine calls them
  plain_grid, plain_degrid   one launch per facet on device buffers
  grid, degrid the batched all-facet passes on a plan that is kept over the major cycles of a chunk
  dirty        a chunk seen once: its plan is built and it is gridded
  cycle        predict, subtract, grid, transform and stitch: one whole major cycle on all facets
  gradient     the chi^2 gradient of a model image (degridding and its adjoint)
  chunk        what comes before gridding: flag preparation, baseline-time sort, BDA map, imaging weights
"""
import functools
import math

import numpy as np
import torch

from ddfacet_amd import _pyGridderSmearPols as gridder
from ddfacet_amd import autograd, bda, chunk, imaging, synth, weights
from ddfacet_amd.cfdev import DeviceCFSet
from ddfacet_amd.cycle import MajorCycle
from ddfacet_amd.facets import DeviceFacetSet
from ddfacet_amd.problems import Facet, Problem, chan_equidistant
from ddfacet_amd.wterm import SpheMachine

C_LIGHT = 299792458.0
FAST = (189, 225, 245, 315, 343, 405, 441, 513, 525, 567, 625, 675, 693, 735, 819, 875, 945, 975)

# What a case holds: the array (antennas in a 20 km disk, or a 1 km core with arms to 8 km), its samples in
# time and frequency, the facets (nfx x nfx of `facet` pixels, padded to `npad`), the CF tables (nw planes of
# supports smin to smax) and the options.  bda: "vis" one block per visibility, "map" the averaging map built
# from the uvw, "uneven" fixed factors by baseline length.
BASE = dict(do="grid", array="disk", nant=27, ntime=100, dt=10.0, nchan=16, f0=1.2e9, f1=1.6e9, nfx=1, facet=405,
            npad=513, cell=2.0, nw=8, smin=7, smax=7, bda="vis", nband=1, stokes="I", jones=0, beam=False,
            decorr=False, precision="mixed")


def case(name=None, **kw):
    c = dict(BASE, **kw)
    if name:
        c["name"] = name
    return c


def listed():
    meerkat = dict(array="meerkat", nant=64, dt=8.0, nchan=64, f0=0.9e9, f1=1.67e9, cell=1.5, nw=32, smax=15,
                   bda="map")
    return [
        # one facet of a short snapshot through the drop-in functions: staging and launch latency
        case("put_snapshot", do="put", ntime=8, npad=513),
        case("get_snapshot_jones", do="get", ntime=20, npad=525, bda="map", jones=1),
        # a whole-field facet, each visibility its own block, on device buffers
        case("plain_grid_facet", do="plain_grid"),
        # facet by facet with averaged blocks and DD Jones matrices
        case("plain_degrid_facets", do="plain_degrid", nfx=3, facet=315, npad=525, nchan=64, bda="map", jones=1),
        # a small field: the smallest whole cycle, where launches and waits are most of the time
        case("cycle_small", do="cycle", nant=7, ntime=10, dt=900.0, nchan=6, nfx=3, facet=81, npad=189, cell=20.0,
             nw=4, smax=9),
        # the wide field, 81 facets with DD Jones: the two directions of the inner loop of imaging
        case("grid_81_jones", do="grid", ntime=150, nfx=9, facet=455, npad=735, jones=1, **meerkat),
        case("degrid_81_jones", do="degrid", ntime=150, nfx=9, facet=455, npad=735, jones=1, **meerkat),
        # all polarisations, beam and DD Jones, decorrelation, in the precision of the reference
        case("grid_iquv_fp64", do="grid", nfx=3, facet=315, npad=525, nchan=32, nband=2, stokes="IQUV", bda="map",
             smax=9, jones=1, beam=True, decorr=True, precision="fp64"),
        # a chunk that is seen once (a dirty image): the plan is part of the work
        case("dirty_25_jones", do="dirty", ntime=75, nfx=5, facet=455, npad=735, jones=1, **meerkat),
        # many facets, four bands, uneven averaging: a whole cycle with the image side
        case("cycle_121_uneven", do="cycle", nfx=11, facet=567, npad=975, nband=4, bda="uneven"),
        # a gradient step of a model fit
        case("gradient_25", do="gradient", nfx=5, facet=405, npad=693, nchan=32, nband=4),
        # a chunk before it is gridded
        case("chunk_before_gridding", do="chunk", ntime=150, nfx=9, facet=455, npad=735, **meerkat),
    ]


def draw(rng):
    """A case of the same ranges: fields of 1 to 49 facets, short and long chunks, every option."""
    do = rng.choice(["put", "get", "plain_grid", "plain_degrid", "grid", "grid", "degrid", "degrid", "dirty", "cycle",
                     "gradient", "chunk"])
    one = do in ("put", "get")
    nfx = 1 if one else rng.choice([1, 2, 3, 4, 5] if do in ("plain_grid", "plain_degrid") else [1, 2, 3, 4, 5, 6, 7])
    npad = rng.choice(FAST[:12] if nfx > 3 or one else FAST)
    facet = max(45, int(npad / rng.uniform(1.3, 1.8)) // 9 * 9)
    smin = rng.choice([5, 7, 9])
    nant, nchan = rng.randint(5, 40), int(math.exp(rng.uniform(math.log(3), math.log(64))))
    jones = rng.choice([0, 0, 1, 1, 1, 2]) if do != "gradient" else rng.choice([0, 0, 1])
    # visibilities: up to what keeps a case below the largest listed one
    nvis = math.exp(rng.uniform(math.log(2e3), math.log(3e5 if one else 2e7 if do == "chunk" else 2e8 / nfx ** 2)))
    if not one:
        nvis = min(nvis, 4e6 if do == "chunk" else 1.5e6)
    ntime = max(2, min(400, int(nvis / (nant * (nant - 1) / 2 * nchan))))
    return case(do=do, array=rng.choice(["disk", "meerkat"]), nant=nant, ntime=ntime, dt=rng.choice([4.0, 8.0, 10.0, 30.0]),
                nchan=nchan, f0=0.9e9, f1=rng.choice([1.2e9, 1.6e9]), nfx=nfx, facet=facet, npad=npad,
                cell=rng.choice([1.5, 2.0, 3.0]), nw=rng.randint(2, 24), smin=smin, smax=smin + 2 * rng.randint(0, 3),
                bda=rng.choice(["vis", "map", "map", "uneven"]),
                nband=1 if do in ("put", "get") else rng.choice([1, 1, 2, 3]) if nchan >= 3 else 1,
                stokes=rng.choice(["I", "I", "I", "IQUV"]) if do not in ("gradient", "cycle") else "I", jones=jones,
                beam=bool(jones and rng.random() < 0.3), decorr=rng.random() < 0.3 and do != "gradient",
                precision=rng.choice(["mixed", "mixed", "mixed", "fp64", "fp32"]) if do in ("grid", "degrid") else "mixed")


# ---- inputs ----------------------------------------------------------------------------------------
def freqs_of(c):
    return np.linspace(c["f0"], c["f1"], c["nchan"])


def observe(c, ha):
    """uvw, antennas and time index of every row, baseline-time order, hour angle `ha` at mid track."""
    rng = np.random.default_rng(2000)
    enu = synth.layout_disk(c["nant"], 20000.0, rng) if c["array"] == "disk" else synth.layout_meerkat_like(c["nant"], rng)
    lat, dec = (45.0, 45.0) if c["array"] == "disk" else (-30.7, -30.0)
    t = (np.arange(c["ntime"]) - (c["ntime"] - 1) / 2.0) * c["dt"]
    uvw, a0, a1, tidx = synth.earth_rotation_uvw(enu, np.deg2rad(lat), np.deg2rad(dec), t * synth.OMEGA_EARTH + ha)
    # arrays are chosen for the field: baselines that fit the facet's uv grid
    fit = 0.46 / (c["cell"] * synth.ARCSEC) * C_LIGHT / c["f1"]
    uvw *= min(1.0, fit / float(np.abs(uvw[:, :2]).max() * 1.02))
    order = np.lexsort((tidx, a1, a0))
    return np.ascontiguousarray(uvw[order]), a0[order].copy(), a1[order].copy(), tidx[order].copy()


@functools.lru_cache(maxsize=4)
def _wmax(key):
    c = dict(key)
    return 1.02 * max(float(np.abs(observe(c, h)[0][:, 2]).max()) for h in (-0.05, 0.0, 0.05)) + 1e-3


@functools.lru_cache(maxsize=2)
def _facets(key):
    """CF tables of every facet: a program makes them once for a run, whatever the chunk."""
    c = dict(key)
    wmax = _wmax(key)
    freqs = freqs_of(c)
    at = [(i * c["facet"] + c["facet"] // 2 - c["nfx"] * c["facet"] // 2) * c["cell"] * synth.ARCSEC for i in range(c["nfx"])]
    lm = [(x, y) for y in at for x in at]
    sups = [int(s) | 1 for s in np.linspace(c["smin"], c["smax"], c["nw"])]
    cf = DeviceCFSet(lm, c["npad"], c["cell"], freqs, c["nw"], sups, 11, wmax)
    sphe = np.float32(SpheMachine(support=c["smin"]).make_sphe(c["npad"])[2].real)
    winfos = np.array([C_LIGHT / freqs[-1], wmax, c["nw"], 11], np.float64)
    data = cf.data.cpu().numpy()
    plane = lambda f, k: data[f, cf.offsets[k]:][:(sups[k % c["nw"]] * 11) ** 2].reshape((sups[k % c["nw"]] * 11,) * 2)  # noqa: E731
    return [Facet(l0=lm[f][0], m0=lm[f][1], cu=float(cf.cu[f]), cv=float(cf.cv[f]),
                  wplanes=[plane(f, k) for k in range(c["nw"])],
                  wplanes_conj=[plane(f, k + c["nw"]) for k in range(c["nw"])], winfos=winfos, sphe=sphe, kms_dir=f,
                  beam_dir=f) for f in range(len(lm))]


@functools.lru_cache(maxsize=2)
def _geometry(nfx, facet, npad, cell):
    g = imaging.FacetGeometry(nfx * facet, nfx, facet, npad, cell * synth.ARCSEC)
    g.spatial_weights()
    return g


def geometry(c):
    return _geometry(c["nfx"], c["facet"], c["npad"], c["cell"])


def key_of(c):
    drop = ("name", "do", "bda", "nband", "stokes", "jones", "beam", "decorr", "precision")
    return tuple(sorted((k, v) for k, v in c.items() if k not in drop))


def block_map(c, uvw, a0, a1, freqs, chan_map):
    if c["bda"] == "vis":
        return bda.bda_map_per_visibility(a0, a1, c["nchan"])
    if c["bda"] == "map":
        return bda.bda_map_device(uvw, a0, a1, freqs, float(freqs[1] - freqs[0]), 0.02, c["cell"] * synth.ARCSEC,
                                  c["facet"], chan_map).cpu().numpy()
    length, code = np.hypot(uvw[:, 0], uvw[:, 1]), a0 * 4096 + a1
    base, inv = np.unique(code, return_inverse=True)
    mean = np.bincount(inv, length) / np.bincount(inv)
    cut = np.quantile(mean, [0.2, 0.4, 0.6, 0.8])
    fac = {"%d:%d" % (k // 4096, k % 4096): (16, 8, 4, 2, 1)[int(np.searchsorted(cut, x, side="right"))]
           for k, x in zip(base.tolist(), mean.tolist())}
    return bda.bda_map_factors(a0, a1, c["nchan"], lambda k: (fac[k], fac[k]), chan_map=chan_map)


def observed(c, seed):
    """uvw, a0, a1, tidx, visibilities (device), flags, weights: point sources and noise, 1 % flagged."""
    rng = np.random.default_rng(seed)
    # (the block map is an output of "chunk": its length is that of one hour angle)
    uvw, a0, a1, tidx = observe(c, rng.uniform(-0.05, 0.05) if c["do"] != "chunk" else 0.0)
    freqs = freqs_of(c)
    nsrc, half = 6, 0.45 * c["nfx"] * c["facet"] * c["cell"] * synth.ARCSEC
    vis = synth.predict_point_sources(uvw, freqs, synth.sky_loguniform(nsrc, half, rng), device="cuda",
                                      chunk_rows=max(1, int(2e7) // (nsrc * c["nchan"])))
    gen = torch.Generator(device="cuda").manual_seed(seed)
    vis += 0.05 * torch.randn(vis.shape, generator=gen, device="cuda", dtype=torch.complex64)
    flags = torch.rand(vis.shape[:2], generator=gen, device="cuda") < 0.01
    flags = flags[:, :, None].expand(vis.shape).contiguous().cpu().numpy()
    w = (0.5 + torch.rand(vis.shape[:2], generator=gen, device="cuda")).cpu().numpy()
    return uvw, a0, a1, tidx, vis, flags, w


def problem(c, seed, host=False):
    uvw, a0, a1, tidx, vis, flags, w = observed(c, seed)
    freqs, nchan = freqs_of(c), c["nchan"]
    facets = _facets(key_of(c))
    chan_map = (np.arange(nchan) * c["nband"] // nchan).astype(np.int32)
    bmap = block_map(c, uvw, a0, a1, freqs, chan_map)
    jones = None
    if c["jones"]:
        nt, nch = min(8, c["ntime"]), min(8, nchan)
        jones = dict(mode=c["jones"], interp=0, apply_amp=1, apply_phase=1, scale=0, calib_error=0.0,
                     kms=synth.random_jones(nt, len(facets), c["nant"], nch, seed + 4),
                     kms_time=(tidx * nt // c["ntime"]).astype(np.int32),
                     kms_chan=(np.arange(nchan) * nch // nchan).astype(np.int32))
        if c["beam"]:
            jones.update(beam=synth.random_jones(2, len(facets), c["nant"], 1, seed + 5, 0.02, 0.1),
                         beam_time=(tidx * 2 // c["ntime"]).astype(np.int32), beam_chan=np.zeros(nchan, np.int32))
    dec = None
    if c["decorr"]:
        duvw = np.cross(np.array([0.0, 0.7, 0.7]), uvw) * synth.OMEGA_EARTH
        dec = (np.ascontiguousarray(duvw), float(c["dt"]), float(freqs[1] - freqs[0]), 1, 1)
    cell = c["cell"] * synth.ARCSEC
    return Problem(uvw=uvw, vis=vis.cpu().numpy() if host else vis, flags=flags, weights=w, freqs=freqs, a0=a0, a1=a1,
                   chan_map=chan_map, chan_map_degrid=chan_map.copy(), bda_grid=bmap, bda_degrid=bmap, facets=facets,
                   npix=c["npad"], nband=c["nband"], npol=len(c["stokes"]), incr=np.array([-cell, cell]),
                   corr_codes=[9, 10, 11, 12], stokes_codes=[1, 2, 3, 4][:len(c["stokes"])], jones=jones, decorr=dec,
                   extra=dict(equidistant=chan_equidistant(freqs)))


def model_image(c, seed, shape):
    """A clean-component image: a few tens of point sources a facet."""
    gen = torch.Generator(device="cuda").manual_seed(seed + 7)
    x = torch.rand(shape, generator=gen, device="cuda")
    return torch.where(x < 30.0 / (c["facet"] ** 2), torch.rand(shape, generator=gen, device="cuda"), torch.zeros(()).cuda())


def model_grids(c, seed, nf):
    """Facet model grids: the transforms of each facet's components, at the scale predict leaves them."""
    n, out = c["npad"], []
    for f in range(nf):
        x = model_image(c, seed + 100 * f, (c["nband"], len(c["stokes"]), n, n))
        out.append(torch.fft.fftshift(torch.fft.fft2(torch.fft.ifftshift(x, dim=(-2, -1))), dim=(-2, -1)) * 11.0 ** 2)
    return torch.stack(out).to(torch.complex64).contiguous()


# ---- prepare ---------------------------------------------------------------------------------------
def prepare(c, seed):
    do, s = c["do"], {"do": c["do"], "case": c}
    if do in ("put", "get"):
        P = problem(c, seed, host=True)
        s.update(P=P, grid=P.new_grid())
        if do == "get":
            s["grid"] = model_grids(c, seed, 1)[0].cpu().numpy()
    elif do == "chunk":
        uvw, a0, a1, tidx, vis, flags, w = observed(c, seed)
        order = np.random.default_rng(seed + 1).permutation(len(a0))
        order = order[np.argsort(tidx[order], kind="stable")]  # time order, as an MS holds the rows
        up = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
        s.update(uvw=up(uvw[order]), a0=up(a0[order]), a1=up(a1[order]), times=up(tidx[order] * c["dt"]),
                 vis=vis[up(order)], flags=up(flags[order].view(np.uint8)), weights=up(w[order]), freqs=freqs_of(c),
                 chan_map=up((np.arange(c["nchan"]) * c["nband"] // c["nchan"]).astype(np.int32)),
                 uvmax=float(np.abs(uvw[:, :2]).max() * c["f1"] / C_LIGHT))
    elif do in ("cycle", "gradient"):
        P = problem(c, seed)
        g = geometry(c)
        m = MajorCycle(P, g, precision=c["precision"])
        image = model_image(c, seed, (c["nband"], len(c["stokes"]), g.m, g.m))
        s.update(cycle=m, image=image, residual=torch.empty_like(m.fs.t["vis"]))
        if do == "gradient":
            s.update(op=autograd.DegridOperator(m), weights=m.fs.t["weights"])
    else:
        P = problem(c, seed)
        fs = DeviceFacetSet(P, with_model=True)
        s["fs"] = fs
        if do in ("degrid", "plain_degrid"):
            fs.models.copy_(model_grids(c, seed, fs.nf))
            s["residual"] = torch.empty_like(fs.t["vis"])
        if do in ("grid", "degrid"):
            fs.plan_batched(precision=c["precision"])
    return s


# ---- run -------------------------------------------------------------------------------------------
def sums(fs):
    return [fs.sumwt] + ([fs.sum_jones, fs.sum_jones_chan] if fs.jones is not None else [])


def run(s):
    do, c = s["do"], s["case"]
    if do == "put":
        P, grid = s["P"], s["grid"]
        grid[...] = 0
        sumwt = np.zeros((P.nband, P.npol))
        sj, sjc = np.zeros((2, P.nband)), np.zeros((2, P.freqs.size))
        gridder.pyGridderWPol32(*P.grid_args(0, grid, sumwt, sum_jones=sj, sum_jones_chan=sjc))
        return [grid, sumwt] + ([sj, sjc] if P.jones is not None else [])
    if do == "get":
        return [gridder.pyDeGridderWPol(*s["P"].degrid_args(0, s["grid"], s["P"].vis.copy()))]
    if do == "chunk":
        return run_chunk(s, c)
    if do == "cycle":
        m = s["cycle"]
        s["residual"].copy_(m.fs.t["vis"])
        return [m.cycle(s["image"], vis=s["residual"]), s["residual"]] + sums(m.fs)
    if do == "gradient":
        x = s["image"].clone().requires_grad_(True)
        loss = autograd.chi2(x, s["op"], s["cycle"].fs.t["vis"], s["weights"])
        loss.backward()
        return [loss.detach(), x.grad]
    fs = s["fs"]
    if do in ("degrid", "plain_degrid"):
        s["residual"].copy_(fs.t["vis"])
        (fs.degrid_batched if do == "degrid" else fs.degrid_plain)(vis=s["residual"])
        return [s["residual"]]
    if do == "dirty":
        fs.plan_batched(precision=c["precision"])
    fs.zero_grids()
    (fs.grid_plain if do == "plain_grid" else fs.grid_batched)()
    return [fs.grids] + sums(fs)


def run_chunk(s, c):
    """Sort a chunk by baseline and time, prepare its flags, build its block map and its imaging weights."""
    index = chunk.sort_baseline_time(s["a0"], s["a1"], s["times"])
    d = chunk.apply_sort(index, {k: s[k] for k in ("uvw", "a0", "a1", "vis", "flags", "weights")})
    frac, _ = chunk.update_flags(d["flags"], d["uvw"], d["vis"], d["a0"], d["a1"], na=c["nant"])
    dfreq = float(s["freqs"][1] - s["freqs"][0])
    bmap = bda.bda_map_device(d["uvw"], d["a0"], d["a1"], s["freqs"], dfreq, 0.02, c["cell"] * synth.ARCSEC, c["facet"],
                              s["chan_map"], na=c["nant"])
    w = weights.imaging_weights(d["uvw"], d["weights"], s["freqs"], uv_cell(c), s["uvmax"])
    return [index, d["flags"], frac, bmap, w]


def uv_cell(c):
    return 1.0 / (c["nfx"] * c["facet"] * c["cell"] * synth.ARCSEC)


def work(c):
    """Inputs read once, outputs written once; the arithmetic of a phased, Jones-corrected sum per
    visibility and facet and of a stamp per block and facet."""
    nrow, nf, npol = c["nant"] * (c["nant"] - 1) // 2 * c["ntime"], c["nfx"] ** 2, len(c["stokes"])
    nvis = nrow * c["nchan"]
    grids = nf * c["nband"] * npol * c["npad"] ** 2 * 8
    cf = nf * sum((11 * (int(x) | 1)) ** 2 for x in np.linspace(c["smin"], c["smax"], c["nw"])) * 2 * 8
    pair = nvis * nf * (16 * 2 + 20) + nvis * nf / (1 if c["bda"] == "vis" else 8) * npol * c["smax"] ** 2 * 8
    do = c["do"]
    if do == "chunk":
        return {"bytes": float(nvis * (32 * 2 + 4 * 2 + 4 * 2) + nrow * 40), "flops": float(nvis * 20)}
    image = (c["nfx"] * c["facet"]) ** 2 * c["nband"] * npol * 4
    fft = 10 * nf * c["nband"] * npol * c["npad"] ** 2 * math.log2(c["npad"])
    grid, degrid = nvis * 40 + nrow * 24 + cf + grids, nvis * 64 + nrow * 24 + cf + grids
    if do in ("cycle", "gradient"):
        return {"bytes": float(grid + degrid + 2 * image), "flops": float(2 * pair + 2 * fft)}
    return {"bytes": float(degrid if do in ("get", "degrid", "plain_degrid") else grid), "flops": float(pair)}


# ---- the same in 64 bits ---------------------------------------------------------------------------
def mul2(*m):
    """The product of 2 x 2 matrices [..., 2, 2]."""
    x = m[0]
    for y in m[1:]:
        x = (x[..., :, :1] * y[..., :1, :]) + (x[..., :, 1:] * y[..., 1:, :])
    return x


class Exact:
    """The gridder, the degridder and its adjoint on the device in complex128, a facet at a time."""

    def __init__(self, P):
        self.P, d = P, "cuda"
        up = lambda x, t=None: torch.as_tensor(np.asarray(x), dtype=t, device=d)  # noqa: E731
        self.uvw, self.freqs = up(P.uvw), up(P.freqs)
        self.vis = P.vis if isinstance(P.vis, torch.Tensor) else up(P.vis)
        m = P.bda_grid
        nb = bda.nblocks_of(m)
        size = m[2:2 + nb].astype(np.int64)
        first = 2 + nb + np.cumsum(size) - size
        nr = size - 2
        ch0, nch = m[first].astype(np.int64), (m[first + 1] - m[first]).astype(np.int64)
        blk = np.repeat(np.arange(nb), nr)
        rows = m[np.repeat(first + 2 - (np.cumsum(nr) - nr), nr) + np.arange(nr.sum())].astype(np.int64)
        self.nb, self.rows, self.rblk = nb, up(rows), up(blk)
        per = up(nch)[self.rblk]
        k = torch.repeat_interleave(torch.arange(len(rows), device=d), per)
        off = torch.arange(len(k), device=d) - (torch.cumsum(per, 0) - per)[k]
        self.row, self.blk = self.rows[k], self.rblk[k]
        self.chan = up(ch0)[self.blk] + off
        self.band, self.nch, self.ch0 = up(P.chan_map)[up(ch0)].long(), up(nch), up(ch0)
        self.mid = up(m[first + 2 + nr // 2].astype(np.int64))
        self.flag = up(P.flags)[self.row, self.chan, 0].bool()
        self.w = up(P.weights)[self.row, self.chan].double() * ~self.flag
        f0 = P.facets[0]
        self.sup = [int(p.shape[0]) // 11 for p in f0.wplanes]
        p = P.npol
        toI = torch.zeros((4, 4), dtype=torch.complex128, device=d)
        toI[0, 0] = toI[0, 3] = toI[1, 0] = toI[2, 1] = toI[2, 2] = 0.5
        toI[1, 3], toI[3, 1], toI[3, 2] = -0.5, -0.5j, 0.5j
        self.to_stokes, self.to_corr = toI[:p], 2.0 * toI.conj().T[:, :p]
        self.jones = None
        if P.jones is not None:
            j = P.jones
            self.mode, self.jones = j["mode"], {q: up(j[q]) for q in j if isinstance(j[q], np.ndarray)}
            self.a = [up(P.a0).long(), up(P.a1).long()]

    def add(self, values, index, size):
        return torch.zeros((size,) + values.shape[1:], dtype=values.dtype, device="cuda").index_add_(0, index, values)

    def phase(self, f, row, chan):
        n0 = math.sqrt(1 - f.l0 ** 2 - f.m0 ** 2) - 1
        x = self.uvw @ torch.tensor([f.l0, f.m0, n0], dtype=torch.float64, device="cuda")
        a = 2 * math.pi / C_LIGHT * x[row] * self.freqs[chan]
        return torch.polar(torch.ones_like(a), a)

    def pair(self, f, row, chan):
        """The two antennas' Jones matrices of (row, chan), and BB."""
        j, out = self.jones, []
        for a in self.a:
            x = j["kms"][j["kms_time"][row].long(), f.kms_dir, a[row], j["kms_chan"][chan].long()].to(torch.complex128)
            if "beam" in j:
                y = j["beam"][j["beam_time"][row].long(), f.beam_dir, a[row], j["beam_chan"][chan].long()]
                x = mul2(x, y.to(torch.complex128))
            out.append(x)
        p, q = out[0].abs(), out[1].abs()
        return out[0], out[1], ((p[:, 0, 0] * q[:, 0, 0] + p[:, 1, 1] * q[:, 1, 1]) / 2) ** 2

    def decorr(self, f, nu):
        if self.P.decorr is None:
            return torch.ones(self.nb, dtype=torch.float64, device="cuda")
        duvw, dt, dnu, _, _ = self.P.decorr
        g = torch.tensor([f.l0, f.m0, math.sqrt(1 - f.l0 ** 2 - f.m0 ** 2) - 1], dtype=torch.float64, device="cuda")
        a = dnu / C_LIGHT * (self.uvw[self.mid] @ g)
        b = nu / C_LIGHT * (torch.from_numpy(duvw).cuda()[self.mid] @ g) * dt
        return torch.sinc(a) * torch.sinc(b)

    def place(self, f, degrid):
        """Each block's CF plane, cell and sub-kernel, and whether it is on the grid."""
        P, u = self.P, self.uvw
        shifted = torch.stack([u[:, 0] + u[:, 2] * f.cu, u[:, 1] + u[:, 2] * f.cv, u[:, 2]], 1)
        if degrid:
            mean = self.add(shifted[self.rows], self.rblk, self.nb)
            cnt = self.add(torch.ones(len(self.rows), dtype=torch.float64, device="cuda"), self.rblk, self.nb)
            c = torch.cumsum(torch.cat([torch.zeros(1, dtype=torch.float64, device="cuda"), self.freqs]), 0)
            fm = (c[self.ch0 + self.nch] - c[self.ch0]) / self.nch
        else:
            ok = ~self.flag
            cnt = self.add(ok.double(), self.blk, self.nb)
            mean = self.add(shifted[self.row] * ok[:, None], self.blk, self.nb)
            fm = self.add(self.freqs[self.chan] * ok, self.blk, self.nb) / cnt
        mean = mean / cnt[:, None]
        wvl, n = fm / C_LIGHT, P.npix
        info = f.winfos
        iw = torch.round((info[2] - 1) * mean[:, 2].abs() * (info[0] * wvl) / info[1])
        good = (cnt > 0) & (iw < info[2])
        iw = torch.where(good, iw, torch.zeros_like(iw)).long()
        S = torch.tensor(self.sup, device="cuda")[iw]
        half = (S - 1) // 2
        loc, off = [], []
        for k in (0, 1):
            pos = torch.nan_to_num(n * float(P.incr[k]) * mean[:, k] * wvl + n // 2)
            at = torch.round(pos)
            good = good & (at - half >= 0) & (at + half < n)
            loc.append(at.long())
            off.append((torch.round((at - pos) * 11).long() + (S * 11 - 1) // 2 - half * 11).clamp(0, 10))
        return iw + torch.where(mean[:, 2] > 0, 0, 10000), loc, off, good, fm

    def stamps(self, f, degrid, plane, loc, off, good):
        """(blocks, cells [k, S, S], CF values) of every plane that has blocks, some blocks at a time."""
        n, nw = self.P.npix, len(self.sup)
        for k in range(2 * nw):
            iw, pos = k % nw, k < nw
            which = torch.nonzero(good & (plane == iw + (0 if pos else 10000)))[:, 0]
            S = self.sup[iw]
            first = pos != degrid  # get() takes the lists swapped
            cf = torch.as_tensor((f.wplanes if first else f.wplanes_conj)[iw], device="cuda").to(torch.complex128)
            cf = cf.reshape(11, 11, S, S)
            for part in which.split(200000):
                r = torch.arange(S, device="cuda") - (S - 1) // 2
                cell = (loc[1][part][:, None, None] + r[:, None]) * n + loc[0][part][:, None, None] + r
                cell = cell + (self.band[part] * self.P.npol * n * n)[:, None, None]
                yield part, cell, cf[off[1][part], off[0][part]]

    def spread(self, f, st, degrid, at, conj=False):
        """Stokes values [block, npol] through the CFs onto a grid [nband, npol, n, n]."""
        P = self.P
        grid = torch.zeros(P.nband * P.npol * P.npix ** 2, dtype=torch.complex128, device="cuda")
        for part, cell, cf in self.stamps(f, degrid, *at[:4]):
            for ip in range(P.npol):
                v = st[part, ip][:, None, None] * (cf.conj() if conj else cf)
                grid.index_add_(0, (cell + ip * P.npix ** 2).reshape(-1), v.reshape(-1))
        return grid.reshape(P.nband, P.npol, P.npix, P.npix)

    def grid(self, i, vis=None):
        """One facet's grid, sumwt, SumJones and SumJonesChan."""
        P, f = self.P, self.P.facets[i]
        vis = self.vis if vis is None else vis
        at = self.place(f, False)
        live = at[3][self.blk] & (self.w > 0)
        dec = self.decorr(f, float(P.freqs.mean()))
        st = torch.zeros((self.nb, 4), dtype=torch.complex128, device="cuda")
        total = torch.zeros((3, P.uvw.shape[0] * P.freqs.size), dtype=torch.float64, device="cuda")  # w, BB w, w dec^2
        for part in torch.nonzero(live)[:, 0].split(2000000):
            row, chan, blk, w = self.row[part], self.chan[part], self.blk[part], self.w[part]
            v = vis[row, chan].to(torch.complex128) * (self.phase(f, row, chan).conj() * w)[:, None]
            bb = torch.ones_like(w)
            if self.jones is not None and self.mode == 1:
                J0, J1, bb = self.pair(f, row, chan)
                v = mul2(J0.mH, v.reshape(-1, 2, 2), J1).reshape(-1, 4)
            st.index_add_(0, blk, v)
            if self.jones is not None and self.mode == 2:
                bb = self.block_pair(f)[2][blk]
            wd = w * dec[blk] ** 2
            total[:, row * P.freqs.size + chan] = torch.stack([w, bb * wd, wd])
        if self.jones is not None and self.mode == 2:
            J0, J1, _ = self.block_pair(f)
            st = mul2(J0.mH, st.reshape(-1, 2, 2), J1).reshape(-1, 4)
        by_chan = total.view(3, -1, P.freqs.size).sum(1)
        by_band = torch.zeros((3, P.nband), dtype=torch.float64, device="cuda")
        by_band.index_add_(1, torch.as_tensor(P.chan_map, device="cuda").long(), by_chan)  # blocks lie in one band
        out = [self.spread(f, st @ self.to_stokes.T, False, at), by_band[0][:, None].expand(P.nband, P.npol)]
        return out + ([by_band[1:] * P.npol, by_chan[1:] * P.npol] if self.jones is not None else [])

    def block_pair(self, f):
        return self.pair(f, self.mid, (2 * self.ch0 + self.nch) // 2)

    def predict(self, i, model, out):
        """out[row, chan, 4] -= the facet's model visibilities."""
        P, f = self.P, self.P.facets[i]
        at = self.place(f, True)
        flat = model.reshape(-1).to(torch.complex128)
        st = torch.zeros((self.nb, P.npol), dtype=torch.complex128, device="cuda")
        for part, cell, cf in self.stamps(f, True, *at[:4]):
            for ip in range(P.npol):
                st[part, ip] = (flat[cell + ip * P.npix ** 2] * cf).sum((1, 2))
        v = (st @ self.to_corr.T) * self.decorr(f, at[4])[:, None]
        if self.jones is not None and self.mode == 2:
            J0, J1, _ = self.block_pair(f)
            v = mul2(J0, v.reshape(-1, 2, 2), J1.mH).reshape(-1, 4)
        flat_out = out.view(-1, 4)
        for part in torch.arange(len(self.row), device="cuda").split(2000000):
            row, chan, blk = self.row[part], self.chan[part], self.blk[part]
            x = v[blk]
            if self.jones is not None and self.mode == 1:
                J0, J1, _ = self.pair(f, row, chan)
                x = mul2(J0, x.reshape(-1, 2, 2), J1.mH).reshape(-1, 4)
            flat_out.index_add_(0, row * P.freqs.size + chan, -x * self.phase(f, row, chan)[:, None])

    def adjoint(self, i, bar):
        """The facet's grid of D^H bar."""
        f = self.P.facets[i]
        at = self.place(f, True)
        st = torch.zeros((self.nb, 4), dtype=torch.complex128, device="cuda")
        for part in torch.arange(len(self.row), device="cuda").split(2000000):
            row, chan, blk = self.row[part], self.chan[part], self.blk[part]
            x = bar[row, chan] * self.phase(f, row, chan).conj()[:, None]
            if self.jones is not None and self.mode == 1:
                J0, J1, _ = self.pair(f, row, chan)
                x = mul2(J0.mH, x.reshape(-1, 2, 2), J1).reshape(-1, 4)
            st.index_add_(0, blk, x)
        st = st * self.decorr(f, at[4])[:, None]
        return self.spread(f, st @ self.to_corr.conj(), True, at, conj=True)


def shifted_fft(x, inverse):
    """The centred transform of DDFacet: forward divided by n^2, inverse unnormalised."""
    n = x.shape[-1]
    y = torch.fft.ifftshift(x, dim=(-2, -1))
    y = torch.fft.ifft2(y) * n ** 2 if inverse else torch.fft.fft2(y) / n ** 2
    return torch.fft.fftshift(y, dim=(-2, -1))


class ExactImage:
    """The image side in 64 bits: facet boxes, norm, stitch, model cut."""

    def __init__(self, c, P):
        g = geometry(c)
        self.g, self.n, self.m = g, g.n, g.m
        self.sw = torch.from_numpy(g.spatial_weights()).cuda()
        self.sphe = torch.from_numpy(np.float32(P.facets[0].sphe)).cuda().double()
        self.inv = torch.from_numpy(np.float32(1.0 / np.float64(np.float32(P.facets[0].sphe)))).cuda().double()
        self.norm = torch.zeros((self.m, self.m), dtype=torch.float32, device="cuda")
        for f in range(g.nf):
            big, box = self.box(f)
            self.norm[big] += self.sw[f][box]
        self.norm = self.norm.double()

    def box(self, f):
        big, box = [], []
        for k in (0, 1):
            a = self.g.pix[f][k] - self.n // 2
            lo, hi = max(0, a), min(self.m, a + self.n)
            big.append(slice(lo, hi))
            box.append(slice(lo - a, hi - a))
        return tuple(big), tuple(box)

    def flip(self, x):  # a grid plane [i, j] = image [j, n - 1 - i]
        return x.transpose(-2, -1).flip(-2)

    def unflip(self, x):
        return x.flip(-2).transpose(-2, -1)

    def stitch(self, image, f, grid, weight):
        im = shifted_fft(grid, True).real * 11.0 ** 2 * self.inv
        im = torch.where(self.sphe < 1e-3, torch.zeros(()).double().cuda(), im)
        big, box = self.box(f)
        x = self.unflip(im) * self.sw[f].double() / weight[..., None, None]
        image[(Ellipsis,) + big] += x[(Ellipsis,) + box]

    def factor(self):
        return (11.0 * self.n) ** 2

    def cut(self, f, image):
        big, box = self.box(f)
        x = torch.zeros(image.shape[:2] + (self.n, self.n), dtype=torch.float64, device="cuda")
        x[(Ellipsis,) + box] = image.double()[(Ellipsis,) + big] / self.norm[big]
        x = torch.where(self.sphe < 1e-3, torch.zeros(()).double().cuda(), x * self.sw[f].double() / self.sphe)
        return shifted_fft((self.flip(x) * self.factor()).to(torch.complex128), False)

    def cut_adjoint(self, f, bar, out):
        x = self.unflip(shifted_fft(bar, True).real / self.n ** 2) * self.factor() * self.sw[f].double() / self.sphe
        x = torch.where(self.sphe < 1e-3, torch.zeros(()).double().cuda(), x)
        big, box = self.box(f)
        out[(Ellipsis,) + big] += x[(Ellipsis,) + box] / self.norm[big]


def exact(c, seed):
    do, nf = c["do"], c["nfx"] ** 2
    if do == "chunk":
        return None
    pairs = c["nant"] * (c["nant"] - 1) // 2 * c["ntime"] * c["nchan"] * nf
    stamps = pairs / (1 if c["bda"] == "vis" else 8) * len(c["stokes"]) * c["smax"] ** 2
    cost = pairs * (2 if c["jones"] else 1) * (2 if do in ("cycle", "gradient") else 1) + stamps / 8
    if cost > (1.0e10 if do in ("degrid", "plain_degrid") else 3.0e9):
        return None
    P = problem(c, seed, host=do in ("put", "get"))
    E = Exact(P)
    stack = lambda parts: [torch.stack(x) for x in zip(*parts)]  # noqa: E731
    if do == "put":
        return E.grid(0)
    if do in ("plain_grid", "grid", "dirty"):
        return stack([E.grid(i) for i in range(nf)])
    out = E.vis.to(torch.complex128, copy=True)
    if do in ("get", "degrid", "plain_degrid"):
        models = model_grids(c, seed, nf)
        for i in range(nf):
            E.predict(i, models[i], out)
        return [out]
    I = ExactImage(c, P)  # noqa: E741
    image = model_image(c, seed, (c["nband"], len(c["stokes"]), I.m, I.m))
    if do == "gradient":
        out = -out
        for i in range(nf):
            E.predict(i, -I.cut(i, image), out)
        w = torch.from_numpy(P.weights).cuda().double()[..., None]
        grad = torch.zeros(image.shape, dtype=torch.float64, device="cuda")
        for i in range(nf):
            I.cut_adjoint(i, E.adjoint(i, 2.0 * w * out), grad)
        return [(w * out.abs() ** 2).sum(), grad]
    for i in range(nf):
        E.predict(i, I.cut(i, image), out)
    dirty, parts = torch.zeros(image.shape, dtype=torch.float64, device="cuda"), []
    for i in range(nf):
        grid, *rest = E.grid(i, out)
        weight = rest[0]
        if len(rest) > 1:
            weight = weight * torch.sqrt(rest[1][0] / rest[1][1])[:, None]
        I.stitch(dirty, i, grid, weight)
        parts.append(rest)
    return [dirty / I.norm, out] + stack(parts)
