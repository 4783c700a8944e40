"""Which kernel a call takes, as far as the size queries tell (CPU: the queries are host code)."""
import pytest

from kernelbench_harbor_amd import _lib


@pytest.fixture(scope="module")
def lib():
    return _lib.load()


@pytest.mark.parametrize("M", [1, 16, 32, 100, 300])
def test_fp8w_workspace_of_any_block(lib, M):
    """The query answers for any block value, with room for every block that the call accepts."""
    for K, N in ((14336, 4096), (1056, 640)):
        most = max(lib.kbh_fp8w_workspace_bytes(M, N, K, b) for b in (32, 64, 128, 256))
        assert most > 0
        for b in (0, 1, 96, 512):
            assert lib.kbh_fp8w_workspace_bytes(M, N, K, b) == most
