"""Which kernel a call takes, as far as the size queries tell (CPU: the queries are host code)."""
import ctypes

import pytest

from kernelbench_harbor_amd import _lib


@pytest.fixture(scope="module")
def lib():
    return _lib.load()


def _kernel(query, *sizes):
    """(kernel code, K splits) of a kbh_*_kernel query."""
    n = ctypes.c_int()
    return query(*sizes, ctypes.byref(n)), n.value


@pytest.mark.parametrize("M", [1, 16, 32, 100, 300])
def test_fp8w_workspace_of_any_block(lib, M):
    """The query answers for any block value, with room for every block that the call accepts."""
    for K, N in ((14336, 4096), (1056, 640)):
        most = max(lib.kbh_fp8w_workspace_bytes(M, N, K, b) for b in (32, 64, 128, 256))
        assert most > 0
        for b in (0, 1, 96, 512):
            assert lib.kbh_fp8w_workspace_bytes(M, N, K, b) == most


# M, K, N, K splits of the decode kernel's plan (the wide tiles' differs): its grid is resident at
# once, or its second row block is mostly padding
@pytest.mark.parametrize("M,K,N,splits", [(127, 4096, 2048, 8), (127, 2048, 4096, 4), (72, 2560, 4096, 5), (96, 3072, 3072, 6)])
def test_fp8w_decode_kernel_stays(lib, M, K, N, splits):
    assert lib.kbh_fp8w_workspace_bytes(M, N, K, 128) == splits * M * N * 4


# T, D, N: base GEMMs of two workgroups per CU, which the wide tiles run faster, and ones that the decode kernel does
@pytest.mark.parametrize("T,D,N,kernel", [
    (57, 3584, 3584, 64), (33, 3072, 3072, 64), (64, 3072, 3584, 64), (96, 2560, 2560, 128), (127, 2048, 3584, 128), (64, 4096, 4096, _lib.KBH_KERNEL_DECODE),
    (17, 7168, 3584, _lib.KBH_KERNEL_DECODE), (32, 7168, 3584, _lib.KBH_KERNEL_DECODE), (80, 5120, 2048, _lib.KBH_KERNEL_DECODE), (127, 4096, 2048, _lib.KBH_KERNEL_DECODE)])
def test_lora_base_kernel(lib, T, D, N, kernel):
    assert lib.kbh_lora_qgemm_kernel(T, D, N, 128, None) == kernel


# M, K, N: calls that the decode kernel runs faster than the wide tiles (which take scratch here), and
# calls past the line
@pytest.mark.parametrize("M,K,N,wide", [(48, 2048, 1408, False), (127, 4096, 1664, False), (33, 8192, 2432, False), (17, 3584, 14336, False),
                                        (17, 11008, 1024, False), (127, 2048, 8576, True), (64, 18944, 2176, True), (32, 14336, 4096, True),
                                        (32, 6144, 11008, True), (24, 7168, 11008, True)])
def test_w8a8_decode_kernel_stays(lib, M, K, N, wide):
    assert (lib.kbh_w8a8_scratch_bytes(M, N, K) > 0) == wide


@pytest.mark.parametrize("M,K,N", [(17, 3584, 18944), (31, 3584, 18944), (32, 14336, 5504)])
def test_w8a8_wide_from_the_third_round(lib, M, K, N):
    assert lib.kbh_w8a8_kernel(M, N, K, None) == 128


@pytest.mark.parametrize("M,K,N,splits", [(160, 7168, 5120, 7), (160, 14336, 2560, 14), (129, 14336, 2560, 14)])
def test_w8a8_many_uneven_splits(lib, M, K, N, splits):
    """256-row tiles that are mostly padding: even splits, not more and shorter ones."""
    assert lib.kbh_w8a8_scratch_bytes(M, N, K) == splits * M * N * 4


# M, K, N, group, dtype, kernel: K that ends in half an iteration of the wide tiles (the decode kernel ran
# all of these), where the decode kernel's estimate is lower and where it is not
@pytest.mark.parametrize("M,K,N,group,dtype,kernel", [
    (64, 896, 4096, 128, _lib.KBH_F16, _lib.KBH_KERNEL_DECODE), (127, 640, 8192, 128, _lib.KBH_BF16, _lib.KBH_KERNEL_DECODE),
    (33, 1408, 2048, 128, _lib.KBH_F16, _lib.KBH_KERNEL_DECODE), (48, 1152, 4096, 128, _lib.KBH_BF16, _lib.KBH_KERNEL_DECODE),
    (48, 1792, 6144, 256, _lib.KBH_F16, _lib.KBH_KERNEL_DECODE), (96, 2304, 4096, 256, _lib.KBH_F16, _lib.KBH_KERNEL_DECODE),
    (256, 320, 2048, 64, _lib.KBH_F16, _lib.KBH_KERNEL_DECODE), (128, 960, 2048, 64, _lib.KBH_BF16, _lib.KBH_KERNEL_DECODE),
    (256, 2752, 8192, 64, _lib.KBH_F16, 128), (127, 1152, 14336, 128, _lib.KBH_F16, 128), (64, 29568, 8192, 128, _lib.KBH_F16, 64), (128, 640, 8192, 128, _lib.KBH_F16, 128),
    (64, 1024, 4096, 128, _lib.KBH_F16, 64)])
def test_w4a16_decode_kernel_stays(lib, M, K, N, group, dtype, kernel):
    assert lib.kbh_w4a16_kernel(M, N, K, group, dtype, None) == kernel


@pytest.mark.parametrize("M,K,N,group,kernel", [
    (96, 2048, 1408, 128, 129), (128, 4096, 384, 64, 129), (65, 1024, 8064, 128, 129), (100, 1024, 128, 32, 129),
    (96, 2048, 4224, 128, 128), (64, 2048, 1408, 128, 64), (96, 2048, 1280, 128, 128), (129, 2048, 1408, 128, 128)])
def test_w4a16_128_column_tiles(lib, M, K, N, group, kernel):
    """65 to 128 rows of a small layer with N of 128 mod 256."""
    for dtype in (_lib.KBH_F16, _lib.KBH_BF16):
        assert lib.kbh_w4a16_kernel(M, N, K, group, dtype, None) == kernel


# rows, K, N: layers that the streaming kernel ran slower than the decode kernel, and ones it runs faster
@pytest.mark.parametrize("M,K,N,kernel", [
    (1, 8192, 10240, _lib.KBH_KERNEL_DECODE), (16, 8192, 12288, _lib.KBH_KERNEL_DECODE), (1, 14336, 10240, _lib.KBH_KERNEL_DECODE),
    (16, 6144, 14336, _lib.KBH_KERNEL_DECODE), (1, 5120, 18944, _lib.KBH_KERNEL_DECODE), (16, 7168, 13824, _lib.KBH_KERNEL_DECODE),
    (16, 3584, 18944, _lib.KBH_KERNEL_STREAM), (1, 18944, 3584, _lib.KBH_KERNEL_STREAM), (16, 29568, 8192, _lib.KBH_KERNEL_STREAM),
    (16, 11008, 4096, _lib.KBH_KERNEL_STREAM), (17, 3584, 18944, 64), (16, 4096, 14336, _lib.KBH_KERNEL_DECODE)])
def test_fp8w_streaming_kernel(lib, M, K, N, kernel):
    assert lib.kbh_fp8w_kernel(M, N, K, 128, None) == kernel


@pytest.mark.parametrize("T,D,F,E", [(127, 4096, 14336, 8), (500, 4096, 14336, 64), (1000, 4096, 14336, 64), (4000, 7168, 2048, 256)])
def test_ffn_stream_slices_are_bounded(lib, T, D, F, E):
    """Streamed batches: h, at most 64 MiB of slices, and tables of a few words per token and expert."""
    assert lib.kbh_qmoe_ffn_workspace_bytes(T, D, F, E) <= 2 * T * F * 2 + (64 << 20) + 256 * (T + E)


# T, D, N, E, whether K is split (fp32 slices next to the one [2T, N] of outputs)
@pytest.mark.parametrize("T,D,N,E,split", [(1024, 1024, 1024, 8, False), (512, 1024, 1024, 8, False), (192, 1024, 2048, 8, False), (384, 1024, 1024, 16, False),
                                           (1, 2048, 1408, 64, True), (16, 2048, 1408, 60, True), (512, 4096, 1024, 8, True), (256, 4096, 14336, 8, False)])
def test_qmoe_split_only_where_it_pays(lib, T, D, N, E, split):
    slices = lib.kbh_qmoe_workspace_bytes(T, D, N, E) // (2 * T * N * 4)
    assert (slices > 1) == split
