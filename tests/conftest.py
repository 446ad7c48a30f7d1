import gc
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
for p in (ROOT, ROOT / "triton-gated-mlp_amd"):
    if str(p) not in sys.path:
        sys.path.insert(0, str(p))


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an AMD GPU (run on the MI355X box)")


@pytest.fixture(autouse=True)
def _collected_heap(request):
    """Tests that account for device memory start without garbage of earlier ones, which a collection in the
    middle of them would free."""
    if request.node.path.name == "test_zz_no_alloc.py":
        gc.collect()
    yield
