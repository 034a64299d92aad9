import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (HIP device)")


@pytest.fixture(scope="session")
def oracle():
    from oracle import oracle as O

    O.lib()
    return O


@pytest.fixture(scope="session")
def hip_ctx():
    from atrip_amd import hip

    ctx = hip.Context(0)
    yield ctx
    ctx.close()


@pytest.fixture(autouse=True)
def automatic_batch(request):
    """Each test that uses the shared context starts with automatic launch
    sizes, whatever an earlier one left."""
    if "hip_ctx" in request.fixturenames:
        request.getfixturevalue("hip_ctx").set_option("batch", 0)
