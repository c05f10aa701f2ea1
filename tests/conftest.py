import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) GPU")
    config.addinivalue_line("markers", "slow: takes more than a few seconds on the CPU")


@pytest.fixture(autouse=True)
def default_factor_schedule(request):
    """GPU tests start from the library's default factorisation schedule, whatever ran before."""
    if request.node.get_closest_marker("gpu") is not None:
        import torch  # noqa: F401  (its HIP runtime is the process's: loaded before the library)

        from germaine_amd import fdfd
        fdfd.factor_tuning()
    yield
