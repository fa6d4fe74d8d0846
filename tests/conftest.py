import gc
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _p in (ROOT, os.path.dirname(os.path.abspath(__file__))):
    if _p not in sys.path:
        sys.path.insert(0, _p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs through libgenllm_hip.so on the GPU)")


@pytest.fixture(scope="session")
def orc():
    import oracle

    oracle.build()
    return oracle


@pytest.fixture(autouse=True)
def no_cyclic_gc(request):
    """No cyclic garbage collection inside a GPU test.  A collection may start
    at any allocation, and destroying an earlier test's CUDA graph (which waits
    for the device) while this test captures its own aborts the process: what
    earlier tests left is collected here, before the test, and the collector
    stays off until it ends."""
    if "gpu" not in request.keywords:
        yield
        return
    gc.collect()
    gc.disable()
    yield
    gc.enable()
