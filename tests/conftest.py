import os
import sys

import numpy as np
import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if REPO not in sys.path:
    sys.path.insert(0, REPO)

GOLDEN = os.path.join(REPO, "tests", "golden")


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) and the built HIP library")


@pytest.fixture(scope="session")
def oracle():
    from oracle.hako_oracle import Oracle
    return Oracle()


@pytest.fixture(scope="session")
def compiled_reference():
    """Skips where the reference's sources, and so the libraries that oracle/ref.mk builds from them, are absent."""
    from oracle.hako_oracle import REF_LIB, REF_MODEL_LIB, REF_NOFAST_LIB
    for lib in (REF_LIB, REF_MODEL_LIB, REF_NOFAST_LIB):
        if not os.path.exists(lib):
            pytest.skip(f"reference library not built: {os.path.basename(lib)}")


@pytest.fixture(scope="session")
def golden():
    cache = {}

    def load(name):
        if name not in cache:
            with np.load(os.path.join(GOLDEN, name), allow_pickle=False) as z:
                cache[name] = {k: z[k] for k in z.files}
        return cache[name]
    return load


@pytest.fixture(scope="session")
def gpu():
    from hako_amd.gpu import Gpu
    return Gpu(int(os.environ.get("HAKO_DEVICE", "0")))
