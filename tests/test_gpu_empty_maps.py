"""Plans of maps whose blocks hold no visibilities (rows of the chunk that a selection has emptied): gridding adds
nothing, degridding leaves the visibilities as they are, and the other map is not touched by it."""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from ddfacet_amd import bda as bdamod
from ddfacet_amd.facets import DeviceFacetSet
from ddfacet_amd.problems import random_problem
from oracle import cpuref

pytestmark = pytest.mark.gpu


def _empty_blocks(n):
    return bdamod.pack({"0:1": ([2] * n, [0, 4] * n)})


@pytest.mark.parametrize("jones", [None, dict(mode=1)])
@pytest.mark.parametrize("which", ["grid", "degrid", "both"])
def test_blocks_without_visibilities(which, jones):
    P = random_problem(61, nfacet=2, facet_spacing_px=9, jones=jones)
    full = P.bda_grid
    P.bda_grid = _empty_blocks(70) if which != "degrid" else full
    P.bda_degrid = _empty_blocks(70) if which != "grid" else full
    fs = DeviceFacetSet(P, with_model=True)
    fs.models.fill_(1.0)
    info = fs.plan_batched()
    assert (info["degrid_vis"] == 0) == (which != "grid")
    fs.zero_grids()
    fs.grid_batched()
    vis = fs.t["vis"].clone()
    fs.degrid_batched(vis=vis)
    torch.cuda.synchronize()
    if which != "degrid":
        assert torch.count_nonzero(fs.grids) == 0 and torch.count_nonzero(fs.sumwt) == 0
    else:
        g, sw = P.new_grid(), np.zeros((P.nband, P.npol))
        cpuref.grid(*P.grid_args(1, g, sw))
        assert rel_l2(fs.grids[1].cpu().numpy(), g) <= 1e-5
    if which != "grid":
        assert torch.equal(torch.view_as_real(vis), torch.view_as_real(fs.t["vis"]))
    else:
        assert not torch.equal(torch.view_as_real(vis), torch.view_as_real(fs.t["vis"]))
    fs.destroy_plan()
