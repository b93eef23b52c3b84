"""A plan grids with the Jones time, channel and antenna maps as they are at the call: a program that changes them in
place (another solution interval, say) gets the sums of the new maps without a new plan.  Against the CPU oracle; bounds
as in test_gpu_batched.py."""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from ddfacet_amd import bda as bdamod
from ddfacet_amd.facets import DeviceFacetSet
from ddfacet_amd.problems import random_problem
from oracle import cpuref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [dict(), dict(jones=dict(mode=1, beam=True)), dict(ncorr=2, corr_codes=(9, 12), npol=2, stokes_codes=(1, 2)),
                                dict(jones=dict(mode=1, apply_phase=0))])
@pytest.mark.parametrize("factors", [(1, 1), (4, 8), (12, 8)])
def test_maps_changed_in_place(kw, factors):
    kw = dict(kw)
    kw.setdefault("jones", dict(mode=1))
    P = random_problem(83, nfacet=5, facet_spacing_px=9, ntime=12, **kw)
    P.bda_grid = P.bda_degrid = bdamod.bda_map_factors(P.a0, P.a1, P.freqs.size, lambda key: factors, P.chan_map)
    fs = DeviceFacetSet(P, with_model=True)
    fs.plan_batched()
    rng = np.random.default_rng(2)
    nt, _, na, nch = P.jones["kms"].shape[:4]
    new = dict(kms_time=rng.integers(0, nt, P.a0.size).astype(np.int32), kms_chan=rng.integers(0, nch, P.freqs.size).astype(np.int32))
    if "beam" in P.jones:
        new["beam_time"] = rng.integers(0, P.jones["beam"].shape[0], P.a0.size).astype(np.int32)
    for k, x in new.items():
        P.jones[k] = x
        fs.jones[k].copy_(torch.from_numpy(x))
    P.a0 = rng.integers(0, na, P.a0.size).astype(np.int32)
    fs.jones["a0"].copy_(torch.from_numpy(P.a0))
    fs.zero_grids()
    fs.grid_batched()
    torch.cuda.synchronize()
    for fi in (0, 4):
        g, sw = P.new_grid(), np.zeros((P.nband, P.npol))
        sj, sjc = np.zeros((2, P.nband)), np.zeros((2, P.freqs.size))
        cpuref.grid(*P.grid_args(fi, g, sw, sum_jones=sj, sum_jones_chan=sjc))
        assert rel_l2(fs.grids[fi].cpu().numpy(), g) <= 1e-5
        np.testing.assert_allclose(fs.sumwt[fi].cpu().numpy(), sw, rtol=1e-10)
        np.testing.assert_allclose(fs.sum_jones[fi].cpu().numpy(), sj, rtol=1e-10)
        np.testing.assert_allclose(fs.sum_jones_chan[fi].cpu().numpy(), sjc, rtol=1e-10, atol=1e-300)
    fs.destroy_plan()
