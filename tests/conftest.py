import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu)")


@pytest.fixture(scope="session")
def oracle():
    from oracle import binding
    binding.lib()
    return binding


@pytest.fixture(scope="session")
def sess():
    """One device context for the whole GPU session (tests run in one process)."""
    from rknpu2_matmul_open_amd import ops
    s = ops.Session()
    yield s
    s.close()


@pytest.fixture
def one_piece(sess):
    """one_piece(call) -> (what the call returns, the kernels it launched).  While a per-kernel profile is on, a large
    call on host buffers does not go in panels of rows."""
    from rknpu2_matmul_open_amd import ops

    def run(call):
        got = []
        kernels = ops.profile_kernels(sess, lambda: got.append(call()), iters=1, warmup=0)
        return got[0], [name for name, _ in kernels]
    return run
