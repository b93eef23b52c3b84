"""Work items, packs and slots of the batched tile passes: few workgroups taking many packs, one item a
tile, items of one batch of records, more workgroups than packs; tiles smaller and larger than a stamp.
Every layout gives the grids and visibilities of the reference (the bound of test_gpu_batched.py)."""
import numpy as np
import pytest
import torch

from cases import problem
from conftest import rel_l2
from test_gpu_batched import TOL, _facet_set, _golden

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["multifacet", "iquv"])
@pytest.mark.parametrize("workgroups,chunk,tile", [(1, 64, 8), (3, 0, 16), (9, 70, 5), (0, 0, 3), (2000, 64, 16), (0, 100000, 24)])
def test_layouts_of_the_work(name, workgroups, chunk, tile):
    P, G = problem(name), _golden(name)
    fs = _facet_set(P)
    fs.plan_batched(tile=tile, chunk=chunk, workgroups=workgroups)
    for _ in range(2):  # the queues start over
        fs.zero_grids()
        fs.grid_batched()
    vis = fs.t["vis"].clone()
    fs.degrid_batched(vis=vis)
    torch.cuda.synchronize()
    for fi in range(fs.nf):
        ref = G["grid_f%d_psf0" % fi]
        g = fs.grids[fi].cpu().numpy()
        assert rel_l2(g, ref) <= TOL
        assert np.array_equal(g != 0, ref != 0)
    model = sum(P.vis - G["vis_f%d" % fi] for fi in range(fs.nf))
    assert rel_l2(P.vis - vis.cpu().numpy(), model) <= TOL
    fs.destroy_plan()
