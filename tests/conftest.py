import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP path)")


def pytest_collection_modifyitems(items):
    # last: it fails where neither the reference tree nor a program built from it
    # is present, which under -x would keep every test after it from running
    items.sort(key=lambda i: i.path.name == "test_gpu_dropin.py")


@pytest.fixture(scope="session")
def gpu_ctx():
    import se_amd
    ctx = se_amd.Context(0)
    yield ctx
    ctx.close()
