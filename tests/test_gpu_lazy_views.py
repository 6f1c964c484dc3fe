"""Tensors whose negation is still to be done (torch's negative bit) go to the library as their
values, as the clone that these calls once made did."""
import pytest
import torch

import azeban_amd as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_out", [64, 32])
def test_lazily_negated_spectrum(cuda, n_out):
    z = torch.fft.rfft2(torch.randn(2, 64, 64, dtype=torch.float64, generator=torch.Generator().manual_seed(3))).cuda()
    neg = torch._neg_view(z)
    assert neg.is_neg() and neg.is_contiguous()
    assert torch.equal(A.fft_c2r(neg, 64), -A.fft_c2r(z, 64))
    assert torch.equal(A.to_physical(neg, n_out), -A.to_physical(z, n_out))
    both = torch._neg_view(z.conj())
    assert torch.equal(A.fft_c2r(both, 64), -A.fft_c2r(z.conj().resolve_conj(), 64))
