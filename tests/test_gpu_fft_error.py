"""The error of the centred facet FFTs against 64 bits.  Bound: a value is rounded once a stage (2.5e-8 in the mean square
of FP32 mantissas) after a product with a twiddle that is rounded itself (1.7e-8), 3.0e-8 a stage together, which add as
a random walk over the stages of both dimensions: 4e-8 sqrt(stages) is asked for.  (Butterflies in FP32 round some
five times a stage and miss it at all of these lengths.)"""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from oracle import imaging as ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,stages", [(225, 8), (243, 10), (405, 10), (512, 6), (675, 10), (1024, 8)])
@pytest.mark.parametrize("inverse", [0, 1])
def test_error_of_the_transform(n, stages, inverse):
    from ddfacet_amd import imaging
    rng = np.random.default_rng(n)
    a = (rng.standard_normal((2, n, n)) + 1j * rng.standard_normal((2, n, n))).astype(np.complex64)
    t = torch.from_numpy(a).cuda()
    imaging.fft2c(t, inverse, 1.0)
    want = (ref.ifft2c if inverse else ref.fft2c)(a.astype(np.complex128))
    assert rel_l2(t.cpu().numpy(), want) <= 4e-8 * np.sqrt(stages)


# both sides of the lengths where a strip of columns narrows from 16 to 8 (593) and to 4 (1107), and the last length of the
# passes (1950: the next that they would factor goes to rocFFT)
@pytest.mark.parametrize("n", [585, 588, 594, 600, 1100, 1120, 1944, 1950, 1960])
def test_strip_widths(n):
    from ddfacet_amd import imaging
    rng = np.random.default_rng(n)
    a = (rng.standard_normal((2, n, n)) + 1j * rng.standard_normal((2, n, n))).astype(np.complex64)
    t = torch.from_numpy(a).cuda()
    imaging.fft2c(t, 1, 1.0)
    assert rel_l2(t.cpu().numpy(), ref.ifft2c(a.astype(np.complex128))) <= (1e-6 if n > 1950 else 2e-7)
