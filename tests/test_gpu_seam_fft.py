"""The standalone transforms at every built length, ragged batches and both precisions, and
the fused initial-data and output paths, against torch's transforms on the CPU in 64 bits."""
import pytest
import torch

import azeban_amd as A

pytestmark = pytest.mark.gpu

LENGTHS = (16, 32, 48, 64, 96, 128, 192, 256, 384, 512, 768, 1024, 1536)


@pytest.fixture(scope="module")
def cuda():
    if not torch.cuda.is_available():
        pytest.skip("needs a HIP device")


def rel(a, b):
    return float(torch.linalg.vector_norm(a.cpu().to(b.dtype) - b) / torch.linalg.vector_norm(b))


def c2r_ref(x, n, dim):
    """Complex passes over the leading axes, then c2r ignoring Im at k = 0 and n/2."""
    x = x.to(torch.complex128)
    if dim > 1:
        x = torch.fft.ifftn(x, dim=tuple(range(1, dim)), norm="forward")
    x = x.clone()
    x[..., 0] = x[..., 0].real + 0j
    x[..., n // 2] = x[..., n // 2].real + 0j
    return torch.fft.irfft(x, n=n, norm="forward")


# tolerances: one transform's rounding, log2(n^dim) eps with the margin of the other FFT tests
@pytest.mark.parametrize("dtype,tol", [(torch.float64, 1e-14), (torch.float32, 1e-6)])
@pytest.mark.parametrize("n", LENGTHS)
def test_lengths_1d_2d(cuda, n, dtype, tol):
    g = torch.Generator().manual_seed(n)
    # an odd number of lines leaves the last pair with one; 1D batches around one workgroup's lines
    cases = [(1, 1), (1, 2), (1, 2 * max(1, 1536 // n) + 1), (1, 999)]
    if n <= 768:
        cases += [(2, 1), (2, 3)]
    for dim, howmany in cases:
        x = torch.randn((howmany,) + (n,) * dim, generator=g, dtype=torch.float64)
        axes = tuple(range(1, dim + 1))
        ref = torch.fft.rfftn(x.to(dtype).double(), dim=axes)
        assert rel(A.fft_r2c(x.to(dtype).cuda()), ref) <= tol, (dim, howmany)
        # not the spectrum of a real field: the imaginary parts that c2r ignores are set
        cdt = torch.complex128 if dtype == torch.float64 else torch.complex64
        z = (ref + 0.3j * torch.randn(ref.shape, generator=g, dtype=torch.float64)).to(cdt)
        zd = z.cuda()
        assert rel(A.fft_c2r(zd, n), c2r_ref(z, n, dim)) <= tol, (dim, howmany)
        assert torch.equal(zd.cpu(), z)  # the input is left as it is


def test_lazy_conjugate_input(cuda):
    z = torch.fft.rfft(torch.randn(4, 64, dtype=torch.float64))
    assert rel(A.fft_c2r(z.cuda().conj(), 64), c2r_ref(z.conj().resolve_conj(), 64, 1)) <= 1e-14
    z = torch.fft.rfft2(torch.randn(2, 64, 64, dtype=torch.float64))
    assert rel(A.to_physical(z.cuda().conj()), c2r_ref(z.conj().resolve_conj(), 64, 2) / 64**2) <= 1e-14


@pytest.mark.parametrize("dim,n", [(2, n) for n in LENGTHS] + [(3, n) for n in (16, 32, 48, 64, 96, 128, 192)])
def test_initialize_all_lengths(cuda, dim, n):
    """Forward transform with the projection fused into its last pass against the two steps apart."""
    g = torch.Generator().manual_seed(7 * n + dim)
    u = torch.randn((dim,) + (n,) * dim, generator=g, dtype=torch.float64)
    ref = torch.fft.rfftn(u, dim=tuple(range(1, dim + 1)))
    i = torch.arange(n, dtype=torch.float64)
    k = [torch.where(i >= n // 2 + 1, i - n, i)] * (dim - 1) + [torch.arange(n // 2 + 1, dtype=torch.float64)]
    k = torch.meshgrid(*k, indexing="ij")
    k2 = sum(x * x for x in k)
    k2.view(-1)[0] = 1.0
    dot = sum(k[d] * ref[d] for d in range(dim)) / k2
    ref = torch.stack([ref[d] - k[d] * dot for d in range(dim)])
    ref.view(dim, -1)[:, 0] = 0
    got = A.initialize(u)
    # a white-noise field keeps most of its energy through the projection: one transform's
    # rounding plus the projection's
    assert rel(got, ref) <= 2e-14
    assert float(got.view(dim, -1)[:, 0].abs().max()) == 0.0


def test_side_stream_lifetimes(cuda):
    """Calls on another stream than the tensors' own are not waited for: the inputs are dropped at
    once and their memory is asked for again before the results are read."""
    x = torch.randn(3, 256, 256, dtype=torch.float64)
    ref = torch.fft.rfftn(x, dim=(1, 2))
    side = torch.cuda.Stream()
    for _ in range(3):
        xd = x.cuda()
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            h = A.fft_r2c(xd)
            back = A.fft_c2r(h, 256)
        del xd
        junk = [torch.full((3, 256, 256), 7.0, dtype=torch.float64, device="cuda") for _ in range(4)]
        side.synchronize()
        assert rel(h, ref) <= 1e-14
        assert rel(back / 256**2, x) <= 1e-14
        del junk, h, back
