"""The plain kernels with 1 and 8 lanes a block (maps with many blocks; the golden cases have few, which take a
wavefront each), against the CPU oracle: blocks of one visibility, blocks larger and smaller than a group,
a last wavefront that is not full, flagged and sparse blocks, stamps beyond 256 cells, every Jones mode,
several polarisations.  Bounds as in test_gpu_plain.py: 1e-5 in relative L2, weights 1e-10."""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from ddfacet_amd import bda as bdamod
from ddfacet_amd.facets import DeviceFacetSet
from ddfacet_amd.problems import random_problem
from oracle import cpuref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("factors", [(1, 1), (3, 4), (1, 7)])
@pytest.mark.parametrize("kind", ["plain", "jones1", "jones2_beam", "iquv_wide", "sparse_decorr"])
def test_groups(factors, kind):
    kw = dict(nant=9, ntime=61, nchan=41, npix=96, sups=(5, 7, 7))
    if factors != (1, 1):
        kw.update(nant=12, ntime=120, nchan=36)
    if kind == "jones1":
        kw.update(jones=dict(mode=1))
    if kind == "jones2_beam":
        kw.update(jones=dict(mode=2, beam=True))
    if kind == "iquv_wide":
        kw.update(npol=4, stokes_codes=(1, 2, 3, 4), sups=(15, 17, 17))
    if kind == "sparse_decorr":
        kw.update(sparsify=True, decorr=True, nband=2)
    P = random_problem(77, **kw)
    P.bda_grid = P.bda_degrid = bdamod.bda_map_factors(P.a0, P.a1, P.freqs.size, lambda key: factors, P.chan_map)
    n = bdamod.nblocks_of(P.bda_grid)
    if kind == "sparse_decorr":
        P.sparsification = np.random.default_rng(3).random(n) < 0.7
    mean = P.uvw.shape[0] * P.freqs.size // n
    assert n > 5461 and (mean < 4 or 4 <= mean < 48)
    fs = DeviceFacetSet(P)
    fs.zero_grids()
    fs.grid_plain()
    rng = np.random.default_rng(5)
    model = (rng.standard_normal((P.nband, P.npol, P.npix, P.npix)) * (1 + 0.5j)).astype(np.complex64)
    fs.models[0].copy_(torch.from_numpy(model))
    vis = fs.t["vis"].clone()
    fs.degrid_plain(vis=vis)
    torch.cuda.synchronize()
    g, sw = P.new_grid(), np.zeros((P.nband, P.npol))
    cpuref.grid(*P.grid_args(0, g, sw))
    assert rel_l2(fs.grids[0].cpu().numpy(), g) <= 1e-5
    np.testing.assert_allclose(fs.sumwt[0].cpu().numpy(), sw, rtol=1e-10)
    want = P.vis.copy()
    cpuref.degrid(*P.degrid_args(0, model, want))
    assert rel_l2(P.vis - vis.cpu().numpy(), P.vis - want) <= 1e-5
