"""Result slots shared by the reductions that return to the host: a slot is free again only when
the work that writes to it has ended."""
import ctypes as C
import subprocess
from pathlib import Path

import numpy as np
import pytest
import torch

from azeban_amd import _capi

HERE = Path(__file__).resolve().parent


def test_slots_and_leases(tmp_path):
    exe = tmp_path / "test_slots"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-pthread", str(HERE / "cpp" / "test_slots.cpp"), "-o",
                    str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout + res.stderr


@pytest.mark.gpu
def test_reductions_are_refused_under_capture(cuda):
    """max_norm and energy_spectrum wait for their stream: under capture they are refused before they
    queue anything, more often than there are slots, the graph holds only what was captured
    around them, and later calls give the right results."""
    import azeban_amd as A

    lib = _capi.load()
    x = torch.linspace(-3.0, 2.0, 5000, dtype=torch.float64, device="cuda")
    rng = np.random.default_rng(4)
    u = A.initialize(rng.standard_normal((2, 64, 64)))
    spectrum = A.energy_spectrum(u)
    torch.cuda.synchronize()
    st, graph = C.c_void_p(), C.c_void_p()
    _capi.check(lib.azb_stream_create(C.byref(st)))
    _capi.check(lib.azb_capture_begin(st))
    norm, spec = C.c_double(-1.0), (C.c_double * 33)()
    print("[case] refused under capture", flush=True)
    _capi.check(lib.azb_scale(2.0, C.c_void_p(x.data_ptr()), x.numel(), st))
    for _ in range(20):
        assert lib.azb_max_norm(C.c_void_p(x.data_ptr()), x.numel(), C.byref(norm), st) == _capi.AZB_ERR_HIP
        assert "captured" in lib.azb_last_error().decode()
        assert lib.azb_energy_spectrum(2, 64, C.c_void_p(u.data_ptr()), spec, st) == _capi.AZB_ERR_HIP
    _capi.check(lib.azb_capture_end(st, C.byref(graph)))
    assert norm.value == -1.0 and A.max_norm(x) == 3.0
    for i in range(3):
        _capi.check(lib.azb_graph_launch(graph, st))
        _capi.check(lib.azb_stream_synchronize(st))
        assert A.max_norm(x) == 3.0 * 2 ** (i + 1)
        # sums of one shell's entries by atomics, in any order
        np.testing.assert_allclose(A.energy_spectrum(u), spectrum, rtol=1e-13)
    _capi.check(lib.azb_graph_destroy(graph))
    _capi.check(lib.azb_stream_destroy(st))


def _mappings():
    with open("/proc/self/maps") as f:
        return sum(1 for _ in f)


@pytest.mark.gpu
@pytest.mark.parametrize("dim", [2, 3])
def test_first_calls_of_a_new_solver_allocate_nothing(cuda, dim):
    """A solver's first step and its first run take as long as the later ones: what they return goes
    through memory that is there.  A pinned allocation shows as a mapping of its own."""
    import math

    import azeban_amd as A

    g = A.Grid(dim, 64)
    rng = np.random.default_rng(5)
    u = A.initialize(rng.standard_normal((dim,) + (64,) * dim))
    grown = []
    for i in range(4):  # the first solver warms the process up
        eq = A.IncompressibleEuler(g, A.SmoothCutoff1D(0.05 / 64, 1.0, 2 * math.pi * 16))
        step = A.SSP_RK3(u.shape, eq)
        sim = A.Simulation(g, 0.2, step, u)
        v = u.clone()
        torch.cuda.synchronize()
        print(f"[case] dim={dim} solver {i}", flush=True)
        before = _mappings()
        dt = step.integrate(1e6, 1e-3, 0.2, v)
        assert sim.simulate_until(1e6, max_steps=2) == 2
        grown.append(_mappings() - before)
        assert 0 < dt <= 1e-3 and sim.time() > 0
    assert grown[1:] == [0, 0, 0], grown


@pytest.mark.gpu
def test_loop_read_of_more_samples_than_a_slot_holds(cuda):
    """1024 samples are reported through one slot, more are copied: the same times and steps either way."""
    from azeban_amd.ensemble import Ensemble, Group

    import azeban_amd as A

    rng = np.random.default_rng(6)
    one = A.initialize(rng.standard_normal((2, 64, 64)))
    for S in (1024, 1025):
        print(f"[case] {S} samples", flush=True)
        ens = Ensemble([Group(2, 64, one.unsqueeze(0).repeat(S, 1, 1, 1), "fp64")], 0.2)
        res = ens.run(1e6, steps_per_launch=2, max_launches=1)
        t = ens.times()[0]
        assert res["steps"] == [[2] * S] and len(set(t)) == 1 and t[0] > 0
        ens.close()
