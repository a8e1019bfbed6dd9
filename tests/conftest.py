import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs on the GPU box)")


def pytest_collection_modifyitems(items):
    """The tests on a library linked from the reference's own sources come
    last: where those sources are absent they fail, and a run that stops at the
    first failure has then run everything else."""
    items.sort(key=lambda item: "test_gpu_dropin" in item.nodeid)


@pytest.fixture(scope="session")
def orc():
    """The C restatement (oracle/liboracle.so), built on first use if absent."""
    lib = os.path.join(ROOT, "oracle", "liboracle.so")
    if not os.path.exists(lib):
        subprocess.run(["make", "-C", os.path.join(ROOT, "oracle"), "liboracle.so"], check=True,
                       capture_output=True)
    from oracle.oracle import Oracle
    return Oracle()
