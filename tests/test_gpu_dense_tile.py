"""A small plan whose records lie in a few uv tiles: hundreds of work items add into the same cells, and their sum
must not lose what the items hold.  Against the CPU oracle on an FP64 grid.  Bound: an item adds at most 64 records in FP32,
which leaves sqrt(64 / 3) 3.4e-8 = 1.6e-7 of its own sum, independent from item to item; a value, its phasor and its CF
product round by 3.4e-8 each; so the grid is within 1.5e-7 of FP64 and 2e-7 is asked for (a chain of 500 sums in
FP32 leaves sqrt(500 / 3) 3.4e-8 = 4.4e-7)."""
import ctypes as C

import numpy as np
import pytest
import torch

from conftest import rel_l2
from ddfacet_amd.facets import DeviceFacetSet
from ddfacet_amd.problems import random_problem
from oracle import cpuref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("jones", [None, dict(mode=1)])
def test_many_items_of_one_tile(jones):
    P = random_problem(41, nant=10, ntime=40, nchan=24, bda="pervis", uv_scale=0.12, flag_frac=0.0, npix=64, jones=jones)
    # one source at the phase centre over noise: the records of a tile add up
    P.vis = (1.0 + 0.1 * P.vis).astype(np.complex64)
    fs = DeviceFacetSet(P, with_model=True)
    info = fs.plan_batched()
    assert info["grid_records"] > 40000 and info["grid_items"] > 500
    fs.zero_grids()
    fs.grid_batched()
    torch.cuda.synchronize()
    g = P.new_grid(np.complex128)
    cpuref.grid(*P.grid_args(0, g, np.zeros((P.nband, P.npol))), f64=True)
    assert rel_l2(fs.grids[0].cpu().numpy(), g) <= 2e-7
    fs.destroy_plan()


def _adjoint(fs, bar):
    from ddfacet_amd._lib import check, lib
    from ddfacet_amd.device import stream_handle
    fs.grids.zero_()
    check(lib().ddf_plan_degrid_adjoint(fs._plan, C.c_void_p(bar.data_ptr()), C.c_void_p(stream_handle())))
    torch.cuda.synchronize()
    return fs.grids[0].cpu().numpy().astype(np.complex128)


def test_adjoint_of_one_tile():
    """The adjoint adds its items' tiles to the grid by atomics.  Against the FP64 sum of the adjoints of 64 interleaved
    parts of the visibilities (a record of zeros adds nothing, so a part's sums are a 64th as long).  Bound: some 50
    items of 2048 records a tile, sqrt(50 / 3) 3.4e-8 = 1.4e-7, and the roundings of a value: 2e-7 (500 items of 64 records
    leave 4.4e-7)."""
    P = random_problem(43, nant=10, ntime=60, nchan=32, bda="pervis", uv_scale=0.12, flag_frac=0.0, npix=64)
    fs = DeviceFacetSet(P, with_model=True)
    info = fs.plan_batched()
    assert info["degrid_records"] > 80000
    rng = np.random.default_rng(1)
    bar = (1.0 + 0.1 * (rng.standard_normal(P.vis.shape) + 1j * rng.standard_normal(P.vis.shape))).astype(np.complex64)
    got = _adjoint(fs, torch.from_numpy(bar).cuda())
    want = 0
    for k in range(64):
        part = np.zeros_like(bar)
        part[k::64] = bar[k::64]
        want = want + _adjoint(fs, torch.from_numpy(part).cuda())
    assert rel_l2(got, want) <= 2e-7
    fs.destroy_plan()
