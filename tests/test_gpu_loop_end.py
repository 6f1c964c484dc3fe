"""The end of a run inside a call of several steps: the last step is clamped onto the target and the
call's remaining steps change nothing.  In 2D the row kernels themselves (one per size)
decide that for every step but the first of a call."""
import math

import pytest
import torch

import azeban_amd as A
from azeban_amd import init as I

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32_mixed"])
@pytest.mark.parametrize("dim,N", [(2, 64), (2, 128), (2, 256), (2, 512), (2, 1024), (3, 64)])
def test_target_reached_within_a_call(cuda, dim, N, precision):
    print(f"[case] {dim}D N={N} {precision}", flush=True)
    g = A.Grid(dim, N)
    eq = A.IncompressibleEuler(g, A.SmoothCutoff1D(0.05 / N, 1.0, 2 * math.pi * N / 4), precision)
    step = A.SSP_RK3(g.shape_fourier(dim), eq)
    u = A.initialize(I.double_shear_layer(N, seed=3) if dim == 2 else I.taylor_green_3d(N))
    probe = A.Simulation(g, 0.2, step, u)
    times = []
    for _ in range(3):
        probe.simulate_until(1e6, max_steps=1)
        times.append(probe.time())
    target = 0.5 * (times[1] + times[2])  # 2.5 steps away
    host, dev = A.Simulation(g, 0.2, step, u), A.Simulation(g, 0.2, step, u)
    assert host.simulate_until_host(target) == 3
    assert dev.simulate_until(target, chunk=5) == 3
    assert dev.time() == host.time() == target
    assert torch.equal(dev.u(), host.u())
    # the next run starts from there
    assert dev.simulate_until(times[2], chunk=4) == host.simulate_until_host(times[2]) == 1
    assert dev.time() == host.time() == times[2]
    assert torch.equal(dev.u(), host.u())
