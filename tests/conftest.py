import gc
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run on the GPU box)")
    config.addinivalue_line("markers", "slow: a full-size run that takes a minute or more")


@pytest.fixture(scope="session")
def oracle_lib():
    import oracle
    oracle.build()
    return oracle


@pytest.fixture(autouse=True)
def _no_garbage_under_allocation_counts(request):
    """Tensors that an earlier test left in a reference cycle must not be freed while a test compares allocated bytes."""
    if request.module.__name__.endswith("no_alloc"):
        gc.collect()
    yield
