"""Degrid pass A gives a record's value to the bit whatever the size of its workgroups: by default one wavefront a
workgroup where only so every work item has a workgroup of its own, and four where the number of workgroups is
asked for. Against the CPU oracle at 1e-5 (relative L2) as well."""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from ddfacet_amd.facets import DeviceFacetSet
from ddfacet_amd.problems import random_problem
from oracle import cpuref

pytestmark = pytest.mark.gpu


# work items: fewer than 2048 (four wavefronts either way), 2048 to 8192 (one by default), more (four)
@pytest.mark.parametrize("nfacet,items", [(1, (1, 2048)), (5, (2049, 8192)), (24, (8193, 1 << 30))])
@pytest.mark.parametrize("precision", ["mixed", "fp64"])
def test_one_and_four_wavefronts(nfacet, items, precision):
    P = random_problem(31, nant=14, ntime=30, nchan=12, npix=513, cell_arcsec=4.0, nfacet=nfacet, uv_scale=0.9)
    rng = np.random.default_rng(8)
    fs = DeviceFacetSet(P, with_model=True)
    m = (rng.standard_normal(tuple(fs.models.shape)) * (1 + 0.5j)).astype(np.complex64)
    fs.models.copy_(torch.from_numpy(m))
    out = []
    for workgroups in (0, 700):
        info = fs.plan_batched(precision=precision, workgroups=workgroups)
        assert items[0] <= info["degrid_items"] <= items[1]
        vis = torch.zeros(P.vis.shape, dtype=torch.complex64, device="cuda")
        for _ in range(2):
            vis.zero_()
            fs.degrid_batched(vis=vis)
            torch.cuda.synchronize()
            out.append(vis.cpu().numpy())
        fs.destroy_plan()
    assert np.abs(out[0]).max() > 0
    for x in out[1:]:
        assert np.array_equal(out[0].view(np.uint32), x.view(np.uint32))
    want = np.zeros_like(P.vis)
    for f in range(nfacet):
        cpuref.degrid(*P.degrid_args(f, m[f], want))
    assert rel_l2(out[0], want) <= 1e-5
