import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

GOLDEN = os.path.join(ROOT, "tests", "golden")


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) GPU")
    config.addinivalue_line("markers", "slow: long-running CPU check")


@pytest.fixture(scope="session")
def oracle():
    from oracle.bindings import Oracle
    return Oracle()


@pytest.fixture(scope="session")
def reference_built():
    """Skips the tests that need the reference engine where it is not built (oracle/Makefile builds
    it where the reference's sources are)."""
    from oracle.bindings import REF_SO
    if not os.path.exists(REF_SO):
        pytest.skip("oracle/_ref/libref.so is not built")


@pytest.fixture(scope="session")
def cpg():
    """The product library, initialised on GPU 0 (gpu tests only)."""
    import cachepotato_amd as C
    C.init(0)
    return C


def golden(name):
    import numpy as np
    return np.load(os.path.join(GOLDEN, name), allow_pickle=False)
