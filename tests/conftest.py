import gc
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP library on cuda:0)")


@pytest.fixture(scope="session")
def backend():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import puter_amd
    return puter_amd.Backend()


@pytest.fixture
def no_collection():
    """For tests that capture a graph: a reference cycle of an earlier test (a caught
    exception holds its frame, the frame the graph) that the collector takes apart while a
    stream is capturing destroys that graph there, which the runtime refuses, and torch ends the
    process.  So cycles are collected before the test, and none while it runs."""
    gc.collect()
    gc.disable()
    yield
    gc.enable()
