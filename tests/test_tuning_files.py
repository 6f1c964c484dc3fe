"""Tuning files: which stored choices a solver takes over (the library replaced by a recorder)."""
import ctypes as C
import json

import pytest
import torch

from azeban_amd import solver as S
from azeban_amd._capi import PROF_FAMILIES

NF = len(PROF_FAMILIES)


class Lib:
    """The three plan calls of one solver."""

    def __init__(self, dim):
        self.dim, self.plans, self.tuned = dim, [0] * NF, 0

    def azb_set_plans(self, handle, plans):
        self.plans = list(plans)
        return 0

    def azb_get_plans(self, handle, out):
        for i, p in enumerate(self.plans):
            out[i] = p
        return 0

    def azb_autotune_plans(self, handle, u, reps):
        self.tuned += 1
        self.plans = [0] * NF if self.dim == 2 else [2, 1, 0, 1, 2, 0]
        return 0


@pytest.fixture
def stored(tmp_path, monkeypatch):
    monkeypatch.setattr(S, "_PLANS", {})
    path = tmp_path / "tuning.json"
    path.write_text(json.dumps({"plans": {"2/512/fp64": [1, 0, 0, 0, 2, 0], "3/256/fp64": [1, 1, 0, 1, 1, 0]}}))
    return str(path)


def _ensure(monkeypatch, dim, N, path):
    lib = Lib(dim)
    monkeypatch.setattr(S, "load", lambda: lib)
    return lib, S._ensure_plans(C.c_void_p(1), dim, N, "fp64", torch.zeros(1), 3, path)


def test_2d_plans_of_older_files_do_not_leave_the_fused_path(stored, monkeypatch):
    lib, plans = _ensure(monkeypatch, 2, 512, stored)
    assert plans == [0] * NF and lib.plans == [0] * NF
    # and the file holds that from then on, beside what else was in it
    with open(stored) as f:
        assert json.load(f)["plans"] == {"2/512/fp64": [0] * NF, "3/256/fp64": [1, 1, 0, 1, 1, 0]}
    # other solvers of the process agree
    lib, plans = _ensure(monkeypatch, 2, 512, None)
    assert plans == [0] * NF and lib.tuned == 0


def test_3d_plans_are_taken_from_the_file(stored, monkeypatch):
    lib, plans = _ensure(monkeypatch, 3, 256, stored)
    assert plans == lib.plans == [1, 1, 0, 1, 1, 0] and lib.tuned == 0
