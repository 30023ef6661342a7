import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (HIP device) and the built libnfx.so")
    config.addinivalue_line("markers", "slow: long CPU test")


@pytest.fixture(scope="session")
def oracle_lib():
    import oracle

    oracle.lib()
    return oracle


@pytest.fixture(scope="module", autouse=True)
def own_step_blocks(request):
    """For the modules whose tests count captured step blocks: a library context of their own, and no garbage collection
    between their tests.  The library finds a captured block by its plan, addresses included; a simulation collected
    in between would give its addresses to the next one, which then replays the old block instead of capturing."""
    if request.module.__name__ not in ("test_gpu_plain", "test_gpu_graph_calls"):
        yield
        return
    import gc

    from nofluidx3d_amd import openCL

    if openCL.context is not None:
        openCL.getCommandQueue().finish()
        openCL.context.release()
        openCL.context = None
    gc.collect()
    gc.disable()
    yield
    gc.enable()
    gc.collect()
