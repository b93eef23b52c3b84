"""Maps with a few large blocks among many small ones: with 1 or 8 lanes a block the plain kernels take the large
ones (more than 32 turns of the lanes) in wavefronts of their own. Against the CPU oracle; bounds as in
test_gpu_plain.py: 1e-5 in relative L2, sums 1e-10."""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from ddfacet_amd import bda as bdamod
from ddfacet_amd.facets import DeviceFacetSet
from ddfacet_amd.problems import random_problem
from oracle import cpuref

pytestmark = pytest.mark.gpu

# blocks of the baselines of antenna 0, of the others: a lane a block and blocks of 32 (the last of its own), 33 and
# 600 visibilities, half of the map large, equal blocks; 8 lanes and blocks of 256, 257 to 270 and 1200
MAPS = {
    "one_32": ((4, 8), (2, 3)), "one_33": ((3, 11), (2, 3)), "one_600": ((30, 20), (2, 3)), "one_equal": ((3, 3), (3, 3)),
    "eight_256": ((16, 16), (4, 5)), "eight_270": ((18, 15), (4, 5)), "eight_1200": ((60, 20), (4, 5)), "eight_equal": ((5, 5), (5, 5)),
}


@pytest.mark.parametrize("name", MAPS)
@pytest.mark.parametrize("kind", ["plain", "jones1", "jones2_beam", "iquv_sparse_decorr"])
def test_large_blocks(name, kind):
    kw = dict(nant=16, ntime=126, nchan=60, npix=96, sups=(5, 7, 7))
    if kind == "jones1":
        kw.update(jones=dict(mode=1))
    if kind == "jones2_beam":
        kw.update(jones=dict(mode=2, beam=True))
    if kind == "iquv_sparse_decorr":
        kw.update(npol=4, stokes_codes=(1, 2, 3, 4), sparsify=True, decorr=True, nband=2)
    P = random_problem(93, **kw)
    f0, f1 = MAPS[name]
    P.bda_grid = P.bda_degrid = bdamod.bda_map_factors(P.a0, P.a1, P.freqs.size, lambda key: f0 if key.startswith("0:") else f1,
                                                       P.chan_map)
    n = bdamod.nblocks_of(P.bda_grid)
    mean = P.uvw.shape[0] * P.freqs.size // n
    assert (n >= 65536 and mean <= 10) if name.startswith("one") else (10 < mean < 256 and n >= 4096)
    if kind == "iquv_sparse_decorr":
        P.sparsification = np.random.default_rng(3).random(n) < 0.7
    fs = DeviceFacetSet(P)
    rng = np.random.default_rng(7)
    model = (rng.standard_normal((P.nband, P.npol, P.npix, P.npix)) * (1 + 0.5j)).astype(np.complex64)
    fs.models[0].copy_(torch.from_numpy(model))
    fs.zero_grids()
    fs.grid_plain()
    vis = fs.t["vis"].clone()
    fs.degrid_plain(vis=vis)
    torch.cuda.synchronize()
    g, sw, want = P.new_grid(), np.zeros((P.nband, P.npol)), P.vis.copy()
    sj, sjc = np.zeros((2, P.nband)), np.zeros((2, P.freqs.size))
    cpuref.grid(*P.grid_args(0, g, sw, sum_jones=sj, sum_jones_chan=sjc))
    cpuref.degrid(*P.degrid_args(0, model, want))
    assert rel_l2(fs.grids[0].cpu().numpy(), g) <= 1e-5
    np.testing.assert_allclose(fs.sumwt[0].cpu().numpy(), sw, rtol=1e-10)
    if P.jones is not None:
        np.testing.assert_allclose(fs.sum_jones[0].cpu().numpy(), sj, rtol=1e-10)
        np.testing.assert_allclose(fs.sum_jones_chan[0].cpu().numpy(), sjc, rtol=1e-10)
    assert rel_l2(P.vis - vis.cpu().numpy(), P.vis - want) <= 1e-5
