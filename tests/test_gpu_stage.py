"""2D column stage kernel: every launch shape gives the results of the separate passes.

One sample and a batch of the same grid take different shapes (tile widths, thread splits,
or the separate passes), so a batch that is bit-identical to its samples solved alone
compares them all; the oracle comparison of single solves is in test_gpu_parity.py."""
import math

import pytest
import torch

import azeban_amd as A
from azeban_amd import init as I
from azeban_amd.ensemble import Ensemble, Group

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cuda():
    if not torch.cuda.is_available():
        pytest.skip("needs a HIP device")


def _solver(N, precision):
    g = A.Grid(2, N)
    return g, A.IncompressibleEuler(g, A.SmoothCutoff1D(0.05 / N, 1.0, 2 * math.pi * N / 4), precision)


# batch sizes on both sides of each line of the shape rule: N = 64, 128 have one shape;
# N = 256 widens its tiles from 8 samples; N = 512 has whole-line tiles at 4 and 13, narrow
# ones at 2 (FP64: 8 too; FP32 then runs the separate passes); N = 1024 batches are separate
@pytest.mark.parametrize("precision", ["fp64", "fp32_mixed"])
@pytest.mark.parametrize("N,samples", [(64, 3), (128, 2), (256, 7), (256, 8), (512, 2), (512, 4), (512, 8), (512, 13),
                                       (1024, 2), (1024, 3)])
def test_batch_shapes_bit_identical_to_single(cuda, N, samples, precision):
    u0 = torch.stack([A.initialize(I.double_shear_layer(N, seed=s + 1)) for s in range(samples)])
    ens = Ensemble([Group(2, N, u0.clone(), precision)], 0.2)
    ens.run(1e6, steps_per_launch=2, max_launches=1)
    g, eq = _solver(N, precision)
    for s in (0, samples - 1):
        sim = A.Simulation(g, 0.2, A.SSP_RK3(g.shape_fourier(2), eq), u0[s])
        assert sim.simulate_until(1e6, max_steps=2) == 2
        assert torch.equal(sim.u(), ens.groups[0].u[s]), f"sample {s}"
        assert sim.time() == ens.times()[0][s]
    ens.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32_mixed"])
@pytest.mark.parametrize("N", [64, 256, 512, 1024])
def test_steps_of_one_call_match_single_steps(cuda, N, precision):
    """The stage kernel carries a call's steps through without control kernels (time, clamp and
    max|u| bins are kept by the step kernels themselves): the same states and dt as one
    fixed step per call."""
    u = A.initialize(I.double_shear_layer(N, seed=5))
    g, eq = _solver(N, precision)
    step = A.SSP_RK3(g.shape_fourier(2), eq)
    sim = A.Simulation(g, 0.2, step, u)
    sim.simulate_until(1e6, max_steps=5, chunk=5)
    max_dt = 0.2 * 2.0 / (0.05 / N * (math.pi * N) ** 2)
    t = 0.0
    for _ in range(5):
        t += step.integrate(1e6, max_dt, 0.2, u)
    assert torch.equal(sim.u(), u) and sim.time() == t
    # a step past the target does nothing (the clamp within a call: test_gpu_loop_end.py)
    before = sim.u().clone()
    assert sim.simulate_until(sim.time(), chunk=3) == 0 and torch.equal(sim.u(), before)


@pytest.mark.parametrize("N", [256, 1024])
def test_radix_plan_path_agrees(cuda, N):
    """A solver with other radix plans runs the separate passes: same results to round-off."""
    u = A.initialize(I.double_shear_layer(N, seed=2))
    _, eq = _solver(N, "fp64")
    a, b = torch.empty_like(u), torch.empty_like(u)
    eq.dudt(a, u)
    eq.set_plans([1, 0, 0, 0, 1, 0])
    eq.dudt(b, u)
    # both are within 1e-12 of the oracle (test_gpu_parity.py)
    assert float((a - b).norm() / a.norm()) <= 2e-12
