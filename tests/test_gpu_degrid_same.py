"""Degrid pass B gives the same visibilities to the bit whether a plan takes it in quads of one run or by
visibility: the FP64 loss of a model fit, repeatable to the bit, must not depend on the map's averaging.  One map
is taken both ways: alone its list is short, so its runs are taken as quads; with the single visibilities of other
baselines behind it the list is long and its quads are empty, so all of it goes by visibility.  (The
visibilities of the first tiles of 256 are compared, whose runs and so whose facet batches are the same in both.)"""
import numpy as np
import pytest
import torch

from ddfacet_amd import bda as bdamod
from ddfacet_amd.facets import DeviceFacetSet
from ddfacet_amd.problems import random_problem

pytestmark = pytest.mark.gpu

# averaging of the baselines of antenna 0: runs of one, of a few and of many visibilities; facets: fewer than
# eight, several batches of a length that is and is not a multiple of eight
CASES = {
    "runs_of_five": dict(factors=(1, 5), nfacet=27),
    "runs_of_one": dict(factors=(1, 1), nfacet=9),
    "runs_of_three_jones": dict(factors=(3, 1), nfacet=20, jones=dict(mode=1)),
    "long_runs_jones_beam": dict(factors=(8, 8), nfacet=13, jones=dict(mode=1, beam=True)),
    "whole_blocks_jones2": dict(factors=(40, 32), nfacet=70, jones=dict(mode=2)),
    "iquv_jones_decorr": dict(factors=(2, 3), nfacet=11, npol=4, stokes_codes=(1, 2, 3, 4), jones=dict(mode=1), decorr=True),
    "two_corrs": dict(factors=(1, 4), nfacet=17, ncorr=2, corr_codes=(9, 12), npol=2, stokes_codes=(1, 2), jones=dict(mode=1)),
    "one_corr": dict(factors=(2, 2), nfacet=10, ncorr=1, corr_codes=(1,)),
}


def _degrid(P, models):
    fs = DeviceFacetSet(P, with_model=True)
    fs.models.copy_(models)
    vis = torch.zeros(P.vis.shape, dtype=torch.complex64, device="cuda")
    fs.plan_batched()
    fs.degrid_batched(vis=vis)
    torch.cuda.synchronize()
    fs.destroy_plan()
    return vis.cpu().numpy()


@pytest.mark.parametrize("name", list(CASES))
def test_quads_and_visibilities_agree_to_the_bit(name):
    kw = dict(CASES[name])
    factors = kw.pop("factors")
    P = random_problem(900 + len(name), nant=8, ntime=40, nchan=32, facet_spacing_px=9, **kw)
    full = bdamod.bda_map_factors(P.a0, P.a1, P.freqs.size,
                                  lambda key: factors if key.startswith("0:") else (1, 1), P.chan_map)
    blocks = [[int(c0), int(c1)] + [int(r) for r in rows] for c0, c1, rows in bdamod.iter_blocks(full)]
    first = [b for b in blocks if P.a0[b[2]] == 0]
    rest = [b for b in blocks if P.a0[b[2]] != 0]
    assert len(rest) > 20000
    rng = np.random.default_rng(5)
    shape = (len(P.facets), P.nband, P.npol, P.npix, P.npix)
    models = (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(np.complex64)
    models[3::5] = 0
    models = torch.from_numpy(models)
    got = []
    for part in (first, first + rest):
        P.bda_grid = P.bda_degrid = bdamod.pack({"0": ([len(b) for b in part], [w for b in part for w in b])})
        got.append(_degrid(P, models))
    # whole blocks within the whole tiles of the short list
    ends = np.cumsum([(len(b) - 2) * (b[1] - b[0]) for b in first])
    n = 0
    for b, end in zip(first, ends):
        if end > ends[-1] // 256 * 256:
            break
        x, y = (v[b[2:], b[0]:b[1]] for v in got)
        np.testing.assert_array_equal(x.view(np.uint32), y.view(np.uint32))
        n += np.count_nonzero(x)
    assert n > 1000
