"""Facets gathered onto an image with one plane (tiles of 32 x 32 pixels, 16 x 16 for a smaller image) and with several
(16 x 16): a plane's pixels are the same to the bit however many planes are stitched with it, and equal the oracle's
to FP32 rounding (1e-6)."""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from oracle import imaging as ref
from test_gpu_imaging import _facets, _setup

pytestmark = pytest.mark.gpu


# 40 tiles of 32 on a side with a ragged last one (one plane: large tiles), 39 (small ones)
@pytest.mark.parametrize("m,n", [(1269, 525), (1245, 525)])
@pytest.mark.parametrize("jones", [True, False])
def test_planes_alone_and_together(m, n, jones):
    from ddfacet_amd import imaging
    geom, sw, sphe, inv, dirty, sumwt, sj = _setup(5, m=m, n=n, nband=1, npol=4, jones=jones)
    d = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    norm = torch.zeros((m, m), dtype=torch.float32, device="cuda")
    imaging.facet_norm(geom, d(sw), norm)
    sjd = None if sj is None else d(sj)
    together = torch.zeros((1, 4, m, m), dtype=torch.float32, device="cuda")
    imaging.stitch(geom, d(sphe), d(inv), d(sw), d(dirty), d(sumwt), sjd, norm, together)
    for p in (0, 3):
        alone = torch.zeros((1, 1, m, m), dtype=torch.float32, device="cuda")
        imaging.stitch(geom, d(sphe), d(inv), d(sw), d(dirty[:, :, p:p + 1]), d(sumwt[:, :, p:p + 1]), sjd, norm, alone)
        assert torch.equal(alone[0, 0].view(torch.int32), together[0, p].view(torch.int32))
    facets = _facets(geom, sw, sphe, inv, dirty, sumwt, sj)
    want = ref.facets_to_im(facets, 1, 4, m, ref.facet_norm(_facets(geom, sw, sphe, inv), m))
    got = together.cpu().numpy()
    fin = np.isfinite(want)
    assert np.array_equal(fin, np.isfinite(got))
    assert rel_l2(got[fin], want[fin]) <= 1e-6
