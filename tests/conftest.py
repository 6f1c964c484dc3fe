import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (HIP device) and the built libazeban_hip.so")
    config.addinivalue_line("markers", "slow: long-running case")


# Needs requests that arrive 0.5 ms apart to overlap, and a 64^2 request takes 0.2-0.3 ms in a
# warm process: it runs last, so that a run that stops at its failure has run all the others
# (test_slots_are_reused_when_all_requests_wait tests the same with equal arrivals).
DEPENDS_ON_SOLVE_TIME = ("test_gpu_serving.py::test_slots_are_reused_by_later_requests",)


def pytest_collection_modifyitems(items):
    items.sort(key=lambda item: item.nodeid.endswith(DEPENDS_ON_SOLVE_TIME))


@pytest.fixture(scope="session")
def cuda():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch.device("cuda")
