"""Grid pass A on runs of one Jones key (mixed precision, per-visibility Jones) where its layout can go
wrong, against the CPU oracle: quads of facets that are not full, more quads than a wavefront has, blocks
of more than 64 visibilities, blocks and runs that are flagged whole, more Jones-channel edges than a walk
has segments, facet groups (per-channel sums that fill LDS), one and two correlations, both Jones tables,
decorrelation, the PSF.  Bounds as in test_gpu_batched.py: grids 1e-5 in relative L2, weight and Jones sums
1e-10."""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from ddfacet_amd import bda as bdamod
from ddfacet_amd.facets import DeviceFacetSet
from ddfacet_amd.problems import random_problem
from oracle import cpuref

pytestmark = pytest.mark.gpu

CASES = {
    "one_facet": dict(nfacet=1),
    "three_facets_pervis": dict(nfacet=3, bda="pervis"),
    "many_quads": dict(nfacet=70, nant=4, ntime=4),
    "large_blocks": dict(nfacet=5, ntime=40, nchan=16, factors=(40, 16)),
    "exactly_64": dict(nfacet=4, ntime=16, nchan=8, factors=(8, 8)),
    "flagged": dict(nfacet=6, ntime=12, flag_all=True),
    "jones_edges": dict(nfacet=4, nchan=24, factors=(3, 24), jones_chans=12),
    "groups": dict(nfacet=40, nant=4, ntime=3, nchan=512, factors=(3, 64), npix=32),
    "no_channel_lds": dict(nfacet=9, nant=3, ntime=2, nchan=2048, factors=(2, 256), npix=32),
    "two_corrs_beam": dict(nfacet=5, ncorr=2, corr_codes=(9, 12), npol=2, stokes_codes=(1, 2), beam=True),
    "one_corr": dict(nfacet=2, ncorr=1, corr_codes=(1,)),
    "amp_only_decorr_bands": dict(nfacet=5, nband=2, npol=4, stokes_codes=(1, 2, 3, 4), decorr=True, apply_phase=0),
}


def _problem(seed, factors=None, flag_all=False, jones_chans=None, beam=False, apply_phase=1, **kw):
    kw.setdefault("nfacet", 1)
    P = random_problem(seed, jones=dict(mode=1, beam=beam, apply_phase=apply_phase), facet_spacing_px=9, **kw)
    if factors:
        P.bda_grid = P.bda_degrid = bdamod.bda_map_factors(P.a0, P.a1, P.freqs.size, lambda key: factors, P.chan_map)
    if flag_all:
        P.flags[:] |= ((P.a0 == 0) & (P.a1 == 1))[:, None, None]
        P.flags[::2] = True
    if jones_chans:
        from ddfacet_amd import synth
        k = P.jones["kms"].shape
        P.jones["kms"] = synth.random_jones(k[0], k[1], k[2], jones_chans, seed + 9, 0.2, 0.5)
        P.jones["kms_chan"] = (np.arange(P.freqs.size) * jones_chans // P.freqs.size).astype(np.int32)
    return P


@pytest.mark.parametrize("name", list(CASES))
def test_runs_against_oracle(name):
    P = _problem(400 + len(name), **CASES[name])
    fs = DeviceFacetSet(P, with_model=True)
    fs.plan_batched()
    for psf in (0, 1):
        fs.zero_grids()
        fs.grid_batched(dopsf=psf)
        torch.cuda.synchronize()
        for fi in sorted({0, fs.nf // 2, fs.nf - 1}):
            g, sw = P.new_grid(), np.zeros((P.nband, P.npol))
            sj, sjc = np.zeros((2, P.nband)), np.zeros((2, P.freqs.size))
            cpuref.grid(*P.grid_args(fi, g, sw, dopsf=psf, sum_jones=sj, sum_jones_chan=sjc))
            assert rel_l2(fs.grids[fi].cpu().numpy(), g) <= 1e-5, (fi, psf)
            np.testing.assert_allclose(fs.sumwt[fi].cpu().numpy(), sw, rtol=1e-10)
            np.testing.assert_allclose(fs.sum_jones[fi].cpu().numpy(), sj, rtol=1e-10)
            np.testing.assert_allclose(fs.sum_jones_chan[fi].cpu().numpy(), sjc, rtol=1e-10, atol=1e-300)
    fs.destroy_plan()
