"""Calls at the borders between kernels: what each accepts, and the kernels that only a few shapes
reach, against the oracles."""
import numpy as np
import pytest
import torch

from kernelbench_harbor_amd import _lib

pytestmark = pytest.mark.gpu


def _int8(M, K, N, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randint(-128, 128, (M, K), generator=g, dtype=torch.int8)
    w = torch.randint(-128, 128, (K, N), generator=g, dtype=torch.int8)
    return x, w


# rows and layers whose call takes scratch on the wide tiles
@pytest.mark.parametrize("M,K,N", [(17, 18944, 2176), (32, 9472, 4224), (127, 18944, 1152)])
def test_w8a8_without_scratch(dev, M, K, N):
    """A workspace alone is enough up to 32 rows, and up to 127 where N is no multiple of 256."""
    lib = _lib.load()
    assert lib.kbh_w8a8_scratch_bytes(M, N, K) > 0
    x, w = _int8(M, K, N, seed=M)
    xd, wd = x.to(dev), w.to(dev)
    ws = torch.empty(lib.kbh_w8a8_workspace_bytes(M, N, K), dtype=torch.uint8, device=dev)
    acc = torch.empty(M, N, dtype=torch.int32, device=dev)
    st = torch.cuda.current_stream().cuda_stream
    assert lib.kbh_w8a8_gemm_i32(xd.data_ptr(), wd.data_ptr(), acc.data_ptr(), ws.data_ptr(), ws.numel(),
                                 None, 0, M, N, K, st) == 0
    # exact: |sum| <= K * 2^14 < 2^53
    assert np.array_equal(acc.cpu().numpy().astype(np.float64), x.double().numpy() @ w.double().numpy())
    # too small a workspace is refused as before
    assert lib.kbh_w8a8_gemm_i32(xd.data_ptr(), wd.data_ptr(), acc.data_ptr(), ws.data_ptr(), 256, None, 0,
                                 M, N, K, st) == _lib.KBH_ERR_WORKSPACE
