import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu)")


# files that test the kernels of the very instances they name, on problems small enough for another tile of them
OWN_TILES = {"test_gpu_parity", "test_gpu_phased", "test_gpu_deep", "test_gpu_fuzz", "test_gpu_channels_first", "test_gpu_colsum",
             "test_gpu_direct_epilogue", "test_gpu_splitk_fold"}


@pytest.fixture(autouse=True)
def own_tiles(request):
    if request.module.__name__.rpartition(".")[2] not in OWN_TILES:
        yield
        return
    from heron_amd import backend
    init = backend.Module.__init__
    with pytest.MonkeyPatch.context() as patch:            # (not the test's own, which it may undo)
        patch.setattr(backend.Module, "__init__", lambda self, desc, timeout_s=0.0, own_tiles=True: init(self, desc, timeout_s, own_tiles))
        yield


@pytest.fixture(scope="session")
def hrn():
    """The ctypes backend; GPU tests fail (not skip) when the HIP library is missing."""
    from heron_amd import backend
    backend.lib()
    return backend
