"""Degrid pass B on quads of four visibilities (mixed precision) where its layout can go wrong, against the
CPU oracle: runs of 2 to more than 256 visibilities (quads that are not full, runs over several tiles, tiles of one
run and of 64), fewer and more facets than a group of eight and than a batch, facets without a model, one, two and
four correlations, no Jones, Jones by visibility and by block, both tables, decorrelation; and maps whose runs are too
short for it.  Bound as in test_gpu_batched.py: visibilities 1e-5 in relative L2 of the prediction."""
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
    "one_facet": dict(nfacet=1, jones=1),
    "runs_of_two": dict(nfacet=3, jones=0, factors=(2, 1)),
    "runs_of_three": dict(nfacet=9, jones=1, factors=(1, 3), nchan=9),
    "runs_of_five": dict(nfacet=8, jones=0, factors=(1, 5), nchan=10),
    "too_short": dict(nfacet=2, jones=1, factors=(1, 1), nant=8, ntime=20, nchan=32),
    "many_facets": dict(nfacet=70, jones=1, nant=4, ntime=5),
    "many_facets_long_runs": dict(nfacet=70, jones=0, nant=4, ntime=8, factors=(8, 8)),
    "long_runs": dict(nfacet=5, jones=0, ntime=60, nchan=16, factors=(60, 16)),
    "empty_models": dict(nfacet=20, jones=1, empty=3),
    "jones_edges": dict(nfacet=4, jones=1, nchan=24, factors=(3, 24), jones_chans=5),
    "by_block_beam": dict(nfacet=6, jones=2, beam=True),
    "two_corrs_beam": dict(nfacet=5, jones=1, ncorr=2, corr_codes=(9, 12), npol=2, stokes_codes=(1, 2), beam=True),
    "one_corr": dict(nfacet=11, jones=0, ncorr=1, corr_codes=(1,)),
    "decorr_iquv": dict(nfacet=5, jones=1, npol=4, stokes_codes=(1, 2, 3, 4), decorr=True),
}


def _problem(seed, jones=0, factors=None, jones_chans=None, beam=False, empty=0, **kw):
    P = random_problem(seed, jones=dict(mode=jones, beam=beam) if jones else None, facet_spacing_px=9, **kw)
    if factors:
        P.bda_grid = P.bda_degrid = bdamod.bda_map_factors(P.a0, P.a1, P.freqs.size, lambda key: factors, P.chan_map)
    if jones_chans:
        from ddfacet_amd import synth
        k = P.jones["kms"].shape
        P.jones["kms"] = synth.random_jones(k[0], k[1], k[2], jones_chans, seed + 9, 0.2, 0.5)
        P.jones["kms_chan"] = (np.arange(P.freqs.size) * jones_chans // P.freqs.size).astype(np.int32)
    return P


@pytest.mark.parametrize("name", list(CASES))
def test_quads_against_oracle(name):
    case = dict(CASES[name])
    empty = case.pop("empty", 0)
    P = _problem(700 + len(name), **case)
    fs = DeviceFacetSet(P, with_model=True)
    rng = np.random.default_rng(len(name))
    models = []
    for fi in range(fs.nf):
        m = (rng.standard_normal(tuple(fs.models[fi].shape)) + 1j * rng.standard_normal(tuple(fs.models[fi].shape))).astype(np.complex64)
        if empty and fi % empty:
            m[:] = 0
        models.append(m)
        fs.models[fi].copy_(torch.from_numpy(m))
    vis = torch.zeros(P.vis.shape, dtype=torch.complex64, device="cuda")
    fs.plan_batched()
    fs.degrid_batched(vis=vis)
    torch.cuda.synchronize()
    want = np.zeros(P.vis.shape, np.complex64)
    for fi in range(fs.nf):
        cpuref.degrid(*P.degrid_args(fi, models[fi], want))
    assert rel_l2(vis.cpu().numpy(), want) <= 1e-5
    fs.destroy_plan()


def test_undefined_position_without_a_model():
    """No model anywhere: the visibilities stay as they are, the ones at an undefined position too."""
    P = _problem(31, nfacet=5, jones=1)
    fs = DeviceFacetSet(P, with_model=True)
    for fi in range(fs.nf):
        fs.models[fi].zero_()
    vis = torch.from_numpy(np.ascontiguousarray(P.vis)).cuda()
    before = vis.clone()
    fs.plan_batched()
    fs.t["uvw"][3] = float("nan")
    fs.degrid_batched(vis=vis)
    assert torch.equal(torch.view_as_real(vis), torch.view_as_real(before))
    fs.destroy_plan()
