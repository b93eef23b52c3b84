"""The stitch sends a list of facets from host memory of the call, which a captured graph would read at its replays
when it is gone: it is refused under capture, and the stream and the next eager call are none the worse for it."""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from oracle import imaging as ref
from test_gpu_imaging import _facets, _setup

pytestmark = pytest.mark.gpu


def test_stitch_is_refused_under_capture():
    from ddfacet_amd import imaging
    from ddfacet_amd._lib import DDFError
    geom, sw, sphe, inv, dirty, sumwt, sj = _setup(3, m=63, nfx=3, n=33, nband=1, npol=1)
    d = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    facets = _facets(geom, sw, sphe, inv, dirty, sumwt, sj)
    norm = ref.facet_norm(facets, 63)
    image = torch.zeros((1, 1, 63, 63), device="cuda")
    args = (geom, d(sphe), d(inv), d(sw), d(dirty), d(sumwt), d(sj), d(norm), image)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    x = torch.zeros(4, device="cuda")
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        x.add_(1.0)
        with pytest.raises(DDFError):
            imaging.stitch(*args, stream=side)
    torch.cuda.current_stream().wait_stream(side)
    for _ in range(3):
        g.replay()
        imaging.stitch(*args)
        torch.cuda.synchronize()
    assert x.cpu().tolist() == [3.0] * 4
    want = ref.facets_to_im(facets, 1, 1, 63, norm)
    fin = np.isfinite(want)
    assert rel_l2(image.cpu().numpy()[fin], want[fin]) <= 1e-6
