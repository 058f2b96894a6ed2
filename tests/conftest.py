import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run on the GPU box)")


@pytest.fixture(scope="session")
def device():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


@pytest.fixture(scope="session", autouse=True)
def _product_workspaces():
    """torch's products keep a workspace (128 MB, and 76 for another library) from their first call to
    the end of the process.  Taken here they have segments of their own; taken inside a test they sit
    in the middle of whatever large segment it left, which then cannot be given back, and tests that
    count what still fits find room in it."""
    import torch
    if not torch.cuda.is_available():
        return
    for dtype in (torch.float32, torch.float64, torch.bfloat16):
        x = torch.ones(64, 64, device="cuda", dtype=dtype)
        torch.mm(x, x)
        torch.addmm(x[0], x, x)
    torch.cuda.synchronize()
    del x
    torch.cuda.empty_cache()
