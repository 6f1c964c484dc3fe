"""Right-hand sides of white noise in every stored mode, the Nyquist ones and a k_last = 0 plane
without Hermitian symmetry among them, against the oracle: the divergence of the products and
its Leray projection hold mode by mode."""
import math

import numpy as np
import pytest
import torch

from oracle import azeban_oracle as O

import azeban_amd as A

pytestmark = pytest.mark.gpu


# every row kernel: M = 96 ... 1536 in 2D, 96, 192, 384 in 3D (768 against the oracle in
# test_gpu_parity.py).  Round-off of the transforms and of the projection is a few times
# eps log2(M^dim) <= 6e-15 of the products' size, which is the RHS's size for white noise.
@pytest.mark.parametrize("dim,N", [(2, 64), (2, 128), (2, 256), (2, 512), (2, 1024), (3, 64), (3, 128), (3, 256)])
def test_rhs_of_unsymmetric_white_noise(cuda, dim, N):
    print(f"[case] white noise in every stored mode dim={dim} N={N}", flush=True)
    rng = np.random.default_rng(13)
    shape = (dim,) + (N,) * (dim - 1) + (N // 2 + 1,)
    uh = O.leray(rng.standard_normal(shape) + 1j * rng.standard_normal(shape))
    visc = (0.05 / N, 1.0, 2 * math.pi * N / 4)
    ref = O.IncompressibleEuler(O.Grid(dim, N), O.SmoothCutoff1D(*visc)).dudt(uh)
    eq = A.IncompressibleEuler(A.Grid(dim, N), A.SmoothCutoff1D(*visc), "fp64")
    u = torch.from_numpy(uh).to("cuda")
    out = torch.empty_like(u)
    eq.dudt(out, u)
    got = out.cpu().numpy()
    assert np.linalg.norm((got - ref).ravel()) <= 1e-13 * np.linalg.norm(ref.ravel())
    # every edge of the spectrum by itself
    for edge in [(slice(None), N // 2), (Ellipsis, 0), (Ellipsis, N // 2)]:
        assert np.linalg.norm((got - ref)[edge].ravel()) <= 1e-12 * np.linalg.norm(ref[edge].ravel())
