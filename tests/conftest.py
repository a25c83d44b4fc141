import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu where there is one)")


@pytest.fixture(scope="session")
def lib():
    """The product's C-ABI library, loaded through the package (fails loudly if unbuilt)."""
    import jax_gpt_amd
    return jax_gpt_amd.lib()
