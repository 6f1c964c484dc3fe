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
