"""The passes of the centred facet FFTs and the tiled facet gathers at the sizes where they can go
wrong, against the numpy restatement (oracle/imaging.py) in FP64.

FFT tolerance: each of the at most 2 x 11 stages rounds a value a few times at 6e-8 and the errors
add as a random walk, sqrt(22) 3 6e-8 = 8e-7, so relative L2 <= 1e-6 (2e-6 for a prime factor above
13, which rocFFT takes through longer convolutions).  The gathers form the same FP32 sums in the
same order: 1e-6."""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from oracle import imaging as ref
from test_gpu_imaging import _facets, _setup

pytestmark = pytest.mark.gpu


# one point, one stage, every radix, a strip that is not full, each strip width and its last length
# (16 columns to 602, 8 to 1137, 4 to 2048), the largest length, lengths left to rocFFT
@pytest.mark.parametrize("n", [1, 2, 3, 4, 8, 11, 13, 17, 34, 39, 512, 600, 616, 729, 735, 1120, 1144, 2028, 2048, 2187])
@pytest.mark.parametrize("inverse", [0, 1])
def test_centred_fft_lengths(n, inverse):
    from ddfacet_amd import imaging
    rng = np.random.default_rng(3 * n + inverse)
    planes = 3 if n <= 600 else 1
    a = (rng.standard_normal((planes, n, n)) + 1j * rng.standard_normal((planes, n, n))).astype(np.complex64)
    t = torch.from_numpy(a).cuda()
    imaging.fft2c(t, inverse, 0.5)
    want = (ref.ifft2c(a.astype(np.complex128)) if inverse else ref.fft2c(a.astype(np.complex128))) * 0.5
    assert rel_l2(t.cpu().numpy(), want) <= (2e-6 if n in (17, 34, 2187) else 1e-6)


# more facets than one batch of the tile's list, planes that do not fill the last group, a facet
# size that leaves a partial tile, a padded length outside the passes' factors
@pytest.mark.parametrize("nfx,m,n,nband", [(17, 153, 15, 5), (3, 63, 33, 1), (3, 99, 51, 3)])
def test_gathers_and_cut(nfx, m, n, nband):
    from ddfacet_amd import abi, imaging  # noqa: F401
    geom, sw, sphe, inv, dirty, sumwt, sj = _setup(11, m=m, nfx=nfx, n=n, nband=nband, npol=1)
    d = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    facets = _facets(geom, sw, sphe, inv, dirty, sumwt, sj)
    norm_ref = ref.facet_norm(facets, m)
    norm, dsphe, dsw = d(norm_ref), d(sphe), d(sw)
    image = torch.zeros((nband, 1, m, m), dtype=torch.float32, device="cuda")
    imaging.stitch(geom, dsphe, d(inv), dsw, d(dirty), d(sumwt), d(sj), norm, image)
    want = ref.facets_to_im(facets, nband, 1, m, norm_ref)
    fin = np.isfinite(want)
    assert np.array_equal(fin, np.isfinite(image.cpu().numpy()))
    assert rel_l2(image.cpu().numpy()[fin], want[fin]) <= 1e-6
    x = np.random.default_rng(5).standard_normal((nband, 1, m, m)).astype(np.float32)
    x[-1] = 0
    # planes that do not follow one another in memory
    spread = torch.zeros((geom.nf, 2, nband, 1, n, n), dtype=torch.complex64, device="cuda")
    models = [spread[i, 1] for i in range(geom.nf)]
    imaging.model_to_grid(geom, dsphe, dsw, d(x), norm, models, 11)
    for i in range(0, geom.nf, 7):
        g = ref.model_grid(x, facets[i], norm_ref, 11)
        assert rel_l2(models[i].cpu().numpy(), g) <= 2e-6
    assert torch.count_nonzero(spread[:, 0]) == 0
