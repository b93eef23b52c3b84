"""The centred facet FFTs of more planes than one launch holds threads for (2^32 / 512 strips of columns): every plane
of a small length comes out as in a call of its own."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,planes", [(1, 9000001), (2, 8400000), (3, 4194305)])
def test_planes_beyond_a_launch(n, planes):
    from ddfacet_amd import imaging
    gen = torch.Generator(device="cuda").manual_seed(n)
    a = torch.randn((planes, n, n), generator=gen, device="cuda", dtype=torch.complex64)
    whole = a.clone()
    imaging.fft2c(whole, 1, 0.5)
    for first in (0, 4194303, 4194304, planes - 70):
        part = a[first:first + 70].clone()
        imaging.fft2c(part, 1, 0.5)
        k = part.shape[0]
        assert torch.equal(torch.view_as_real(part), torch.view_as_real(whole[first:first + k]))
