"""Right-hand sides of states with one large velocity component.

The rounding of the large component's square (eps u^2) must stay where its exact value has no
effect: in a flow invariant along its own axis it drops out of the other components'
equations, and in a separable shear layer u = (U(y), f(x)) out of everything.  Both have
references without the products: an invariant flow's in-plane components obey the 2D
equation, and a separable one's only product with an effect is the outer product U f.

Tolerance N * 1e-15: transforms round at eps log2(M^dim) <= 30 eps of the product, in every
mode alike; the derivative weighs that noise with |k| up to 2 pi N / 2, the RHS itself sits at
|k| >= 2 pi 10 or so, so relative errors are up to 30 eps N / 20 = 3.3e-16 N, and a margin of 3.
The large component's ratio must not appear in it, except where it shares a packed
transform with the component compared (see each test)."""
import math

import numpy as np
import pytest
import torch

from oracle import azeban_oracle as O

import azeban_amd as A

pytestmark = pytest.mark.gpu


def _visc(N):
    return (0.05 / N, 1.0, 2 * math.pi * N / 4)


def _rhs(dim, N, u):
    eq = A.IncompressibleEuler(A.Grid(dim, N), A.SmoothCutoff1D(*_visc(N)), "fp64")
    out = torch.empty_like(u)
    eq.dudt(out, u)
    return out


def _norm(a):
    return float(np.linalg.norm(np.asarray(a).ravel()))


def _planar_flow(N, seed):
    """Full 2D spectra of a divergence-free field and a scalar, modes |k| <= 6, rms 1."""
    rng = np.random.default_rng(seed)
    k = np.fft.fftfreq(N, 1.0 / N)
    k1, k2 = k[:, None], k[None, :]
    kk = k1**2 + k2**2
    band = (kk > 0) & (kk <= 36)
    psi, w = (np.where(band, np.fft.fft2(rng.standard_normal((N, N))) / (1 + kk), 0.0) for _ in range(2))
    u = np.stack([1j * k2 * psi, -1j * k1 * psi])
    rms = lambda a: math.sqrt(float((np.abs(a) ** 2).sum())) / N**2
    return u / rms(u), w / rms(w)


# every FP64 row kernel of the 3D path.  The axial component along axis 0 or 1 shares a packed
# transform with an in-plane one, whose rounding is then relative to the axial one's size.
@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("N", [64, 128, 256, 512])
def test_invariant_flow_with_large_axial_velocity(cuda, N, axis):
    print(f"[case] axis-{axis} invariant flow N={N}", flush=True)
    ratio = 100.0
    p, w = _planar_flow(N, 3 + axis)
    nh = N // 2 + 1
    ref = O.IncompressibleEuler(O.Grid(2, N), O.SmoothCutoff1D(*_visc(N))).dudt(p[:, :, :nh].copy())
    u = torch.zeros((3, N, N, nh), dtype=torch.complex128, device="cuda")
    plane = [d for d in range(3) if d != axis]

    def slab(t, c):  # the modes without variation along the axis
        return (t[c, 0], t[c, :, 0], t[c, :, :, 0])[axis]

    for c, f in zip(plane + [axis], [p[0], p[1], ratio * w]):
        full = torch.from_numpy(N * f).to("cuda")
        slab(u, c).copy_(full if axis == 2 else full[:, :nh])
    out = _rhs(3, N, u)
    got = np.stack([slab(out, c).cpu().numpy()[:, :nh] / N for c in plane])
    tol = N * 1e-15 * (1.0 if axis == 2 else ratio)
    for c in range(2):
        assert _norm(got[c] - ref[c]) <= tol * _norm(ref[c]), (c, _norm(got[c] - ref[c]) / _norm(ref[c]))
    # and nothing that varies along the axis
    for c in plane:
        slab(out, c).zero_()
        assert float(out[c].abs().max()) <= tol * N * float(np.abs(ref).max())


# every FP64 row kernel of the 2D path.  Lines along the last axis hold both components packed, so
# where the large one varies along them (U(y), axis "last") only the small one's equation is
# compared; the large one constant along each line (U(x)) leaves both exact.
@pytest.mark.parametrize("axis", ["first", "last"])
@pytest.mark.parametrize("N", [64, 128, 256, 512, 1024])
def test_separable_shear_layer(cuda, N, axis):
    print(f"[case] separable shear layer along the {axis} axis N={N}", flush=True)
    x = np.arange(N) / N
    U = np.tanh(np.where(x <= 0.5, x - 0.25, 0.75 - x) / 0.05)
    f = 1e-4 * (np.sin(2 * np.pi * x) + 0.3 * np.sin(14 * np.pi * x + 1))
    nh = N // 2 + 1
    k = np.fft.fftfreq(N, 1.0 / N)
    big, small = (np.where(np.abs(k) < N // 2, np.fft.fft(a), 0.0) for a in (U, f))
    # component 0 varies along the last axis only, component 1 along the first only
    a, b = (big, small) if axis == "last" else (small, big)
    u = np.zeros((2, N, nh), complex)
    u[0, 0, :] = N * a[:nh]
    u[1, :, 0] = N * b
    u[:, 0, 0] = 0.0
    B12 = u[0, 0, None, :] * u[1, :, 0, None] / N**2
    k1, k2 = 2 * np.pi * k[:, None], 2 * np.pi * np.arange(nh)[None, :]
    kk = k1**2 + k2**2
    b = 1j * np.stack([k2 * B12, k1 * B12])
    div = np.divide(k1 * b[0] + k2 * b[1], kk, out=np.zeros_like(B12), where=kk > 0)
    nu = np.asarray(O.SmoothCutoff1D(*_visc(N)).eval(np.sqrt(kk)))
    ref = -(b - np.stack([k1 * div, k2 * div])) + nu * u
    ref[:, 0, 0] = 0.0
    got = _rhs(2, N, torch.from_numpy(u).to("cuda")).cpu().numpy()
    for c in (0, 1) if axis == "first" else (1,):
        assert _norm(got[c] - ref[c]) <= N * 1e-15 * _norm(ref[c]), (c, _norm(got[c] - ref[c]) / _norm(ref[c]))
