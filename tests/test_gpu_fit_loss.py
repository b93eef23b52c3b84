"""The FP64 loss of a model fit, as numbers: autograd.chi2 and a weighted sum of the model grids, at facet lengths
of every kind of factor.  The loss is FP64 and repeatable to the bit, so a program compares it between runs; the values
were recorded with the models' transforms as one 2-D rocFFT plan and degrid pass B by visibility (MI355X, ROCm 7.2).
Bounds: the degridder and the cut round as they did, so the loss is held to 1e-9, a twentieth of an FP32
rounding; the model grids, summed with random signs in FP64, to 1e-9 of their norm (another transform's rounding
moves that by its error, 3e-8 to 1e-7)."""
import numpy as np
import pytest
import torch

from ddfacet_amd import synth
from ddfacet_amd.problems import Problem, make_cf_facet
from ddfacet_amd import bda as bdamod

pytestmark = pytest.mark.gpu

LENGTHS = {
    33: (124678.16679777813, 0.5956521120425864),
    45: (305026.4729848418, 1.3682372509082246),
    63: (346799.0198652382, 0.46174558959244977),
    81: (813769.1703406386, 0.8641320908032648),
    125: (1063550.545153675, -0.2665492568347568),
    135: (1675007.547610816, -0.6042344835895502),
    189: (2318424.6562169334, -0.17048963114148802),
    243: (5348210.0562473675, -0.40542677067021277),
    245: (5126647.748041679, 0.9116065993114084),
    343: (78829945.15622869, -0.5652289077869349),
    405: (10968126.86773135, -0.43366044757229955),
    513: (34468846.74803297, -0.2702658026473298),
}


def measure(n):
    from ddfacet_amd import autograd, imaging
    from ddfacet_amd.cycle import MajorCycle
    nfx, facet, cell, nchan = 3, (2 * n // 3) | 1, 4.0, 8
    freqs = np.linspace(1.2e9, 1.6e9, nchan)
    geom = imaging.FacetGeometry(nfx * facet, nfx, facet, n, cell * synth.ARCSEC)
    diam = 0.8 * 0.42 / (2 * cell * synth.ARCSEC) * 299792458.0 / 1.6e9
    obs = synth.make_observation("disk", 7, 12, 600.0, freqs, 45.0, -30.7, n, sort_by_baseline=True, diameter_m=diam)
    wmax = float(np.abs(obs.uvw[:, 2]).max()) + 1e-3
    facets = []
    for k, (l, m) in enumerate(geom.lm):
        f = make_cf_facet(l, m, n, cell, freqs, 2, [5, 7], 5, wmax)
        f.kms_dir = k
        facets.append(f)
    rng = np.random.default_rng(n)
    shape = (obs.nrow, nchan, 4)
    vis = (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(np.complex64)
    jones = dict(mode=1, interp=0, apply_amp=1, apply_phase=1, scale=0, calib_error=0.0,
                 kms=synth.random_jones(3, nfx * nfx, 7, 2, n, 0.2, 0.5), kms_time=(obs.tidx // 4).astype(np.int32),
                 kms_chan=(np.arange(nchan) // 4).astype(np.int32))
    cmap = np.zeros(nchan, np.int32)
    bmap = bdamod.bda_map_factors(obs.a0, obs.a1, nchan, lambda k: (2, 4), cmap)
    P = Problem(uvw=obs.uvw, vis=vis, flags=np.zeros(shape, bool), weights=rng.uniform(0.5, 1.5, shape[:2]).astype(np.float32),
                freqs=freqs, a0=obs.a0, a1=obs.a1, chan_map=cmap, chan_map_degrid=cmap.copy(), bda_grid=bmap,
                bda_degrid=bmap, facets=facets, npix=n, nband=1, npol=1,
                incr=np.array([-cell * synth.ARCSEC, cell * synth.ARCSEC]), corr_codes=[9, 10, 11, 12], stokes_codes=[1],
                jones=jones)
    cyc = MajorCycle(P, geom)
    x = np.where(rng.random((1, 1, geom.m, geom.m)) < 0.01, rng.random((1, 1, geom.m, geom.m)), 0).astype(np.float32)
    x = torch.from_numpy(x).cuda()
    loss = autograd.chi2(x, autograd.DegridOperator(cyc), cyc.fs.t["vis"], cyc.fs.t["weights"])
    grids = cyc.fs.models.cpu().numpy().astype(np.complex128)
    sign = rng.choice([-1.0, 1.0], grids.shape)
    cyc.fs.destroy_plan()
    return float(loss), float((grids * sign).sum().real / np.linalg.norm(grids))


@pytest.mark.parametrize("n", list(LENGTHS))
def test_loss_and_model_grids(n):
    loss, grids = measure(n)
    assert abs(loss / LENGTHS[n][0] - 1) <= 1e-9
    assert abs(grids - LENGTHS[n][1]) <= 1e-9
