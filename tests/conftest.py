import os
import sys

# The golden outputs are fp32 sums in the order of OpenBLAS's AVX2 kernels; the AVX-512 kernels that it picks on newer
# CPUs add in another order (up to 2.4e-6 apart, the test allows 1e-6).  Read when numpy is loaded.
os.environ.setdefault("OPENBLAS_CORETYPE", "Haswell")

import pytest  # noqa: E402

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu)")


@pytest.fixture(scope="session")
def device():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")
