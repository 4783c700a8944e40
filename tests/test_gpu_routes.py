"""Calls at the borders between kernels: what each accepts, and the kernels that only a few shapes
reach, against the oracles."""
import numpy as np
import pytest
import torch

from kernelbench_harbor_amd import _lib, inputs, ops
from kernelbench_harbor_amd.harness import compare
from oracle import fp8w as of
from oracle import lora as ol
from oracle import w4a16 as ow

pytestmark = pytest.mark.gpu

F16, BF16 = torch.float16, torch.bfloat16
DT = {F16: _lib.KBH_F16, BF16: _lib.KBH_BF16}


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


# rows, K, N whose W8A8, W4A16 and FP8 calls take slices on the wide tiles and ran without before them
@pytest.mark.parametrize("M,K,N", [(300, 2048, 384), (129, 4096, 640)])
def test_calls_without_scratch(dev, M, K, N):
    """More than 128 rows of N of 128 mod 256 are accepted without scratch (and FP8 calls without a workspace),
    on the LDS-staged kernels; N a multiple of 256 is refused as before (W4A16, W8A8)."""
    lib = _lib.load()
    st = torch.cuda.current_stream().cuda_stream
    assert lib.kbh_w8a8_scratch_bytes(M, N, K) > 0 and lib.kbh_w4a16_scratch_bytes(M, N, K, 128) > 0
    x, w = _int8(M, K, N, seed=M)
    xd, wd = x.to(dev), w.to(dev)
    acc = torch.empty(M, N, dtype=torch.int32, device=dev)
    call = lambda n: lib.kbh_w8a8_gemm_i32(xd.data_ptr(), wd.data_ptr(), acc.data_ptr(), None, 0, None, 0, M, n, K, st)
    assert call(N) == 0
    assert np.array_equal(acc.cpu().numpy().astype(np.float64), x.double().numpy() @ w.double().numpy())
    assert call(256) == _lib.KBH_ERR_WORKSPACE
    x, q, s, z = inputs.w4a16(M, K, N, 128, F16, seed=M)
    d = [t.to(dev) for t in (x, q, s, z)]
    y = torch.empty(M, N, dtype=F16, device=dev)
    call = lambda n: lib.kbh_w4a16_gemm(*[t.data_ptr() for t in d], y.data_ptr(), None, 0, None, 0, M, n, K, 128, 0, st)
    assert call(N) == 0
    cmp = compare(y, ow.forward(x.float().numpy(), q.numpy(), s.float().numpy(), z.float().numpy()))
    assert cmp.ok, cmp
    assert call(256) == _lib.KBH_ERR_WORKSPACE
    x, w, s = inputs.fp8w(M, K, N, 128, F16, seed=M)
    d = [t.to(dev) for t in (x, w, s)]
    assert lib.kbh_fp8w_workspace_bytes(M, N, K, 128) > 0
    assert lib.kbh_fp8w_gemm(*[t.data_ptr() for t in d], y.data_ptr(), None, 0, M, N, K, 128, 0, st) == 0
    cmp = compare(y, of.forward(x.float().numpy(), w.view(torch.uint8).numpy(), s.float().numpy()))
    assert cmp.ok, cmp


def _w4a16(dev, M, K, N, group, dtype, kernel, cols):
    assert _lib.load().kbh_w4a16_kernel(M, N, K, group, DT[dtype], None) == kernel
    x, q, s, z = inputs.w4a16(M, K, N, group, dtype, seed=M + K)
    y = ops.w4a16_gemm(*[t.to(dev) for t in (x, q, s, z)])
    for c in cols:
        w = slice(c.start // 8, c.stop // 8)
        gt = ow.forward(x.float().numpy(), q[:, w].numpy(), s[:, c].float().numpy(), z[:, c].float().numpy())
        cmp = compare(y[:, c], gt)
        assert cmp.ok, cmp


def _fp8w(dev, M, K, N, block, dtype, kernel, cols):
    assert _lib.load().kbh_fp8w_kernel(M, N, K, block, None) == kernel
    x, w, s = inputs.fp8w(M, K, N, block, dtype, seed=M + K)
    y = ops.fp8w_gemm(x.to(dev), w.to(dev), s.to(dev))
    codes = w.view(torch.uint8).numpy()
    for c in cols:
        cmp = compare(y[:, c], of.forward(x.float().numpy(), codes[:, c], s[:, c].float().numpy()))
        assert cmp.ok, cmp


def _w8a8(dev, M, K, N, kernel, cols):
    assert _lib.load().kbh_w8a8_kernel(M, N, K, None) == kernel
    x, w = _int8(M, K, N, seed=M + K)
    acc = ops.w8a8_gemm_i32(x.to(dev), w.to(dev))
    for c in cols:  # exact: |sum| <= K * 2^14 < 2^53
        want = x.double().numpy() @ w[:, c].double().numpy()
        assert np.array_equal(acc[:, c].cpu().numpy().astype(np.float64), want)


# 256-row tiles on the 12-wave kernel: two row blocks, the last column tile overlapping its neighbour
# (the last 512 columns hold the overlap), K that ends in half an iteration, or is one
WIDE256 = (300, 32640)
ENDS = (slice(0, 256), slice(WIDE256[1] - 512, WIDE256[1]))


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("K,group", [(896, 128), (960, 64), (1280, 256), (64, 32), (512, 128)])
def test_256_row_tiles(dev, K, group, dtype):
    M, N = WIDE256
    print(f"[256 rows] K={K} g{group} {dtype}", flush=True)
    _w4a16(dev, M, K, N, group, dtype, 256, ENDS)
    _fp8w(dev, M, K, N, group, dtype, 256, ENDS)


@pytest.mark.parametrize("K", [128, 896, 1408, 512])  # K / 64 of 2 mod 4: half an iteration; whole ones
def test_256_row_tiles_int8(dev, K):
    _w8a8(dev, *(WIDE256[0], K, WIDE256[1]), 256, ENDS)


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("M", [33, 64])
def test_64_row_tiles(dev, M, dtype):
    """Layers whose decode grid is several rounds, or workgroups of one wave."""
    for K, N in ((1408, 2048), (5120, 5120)):
        cols = (slice(0, 256), slice(N - 256, N))
        _fp8w(dev, M, K, N, 128, dtype, 64, cols)
    _w4a16(dev, M, 2048, 2432, 128, dtype, 64, (slice(0, 256), slice(2432 - 512, 2432)))


# The LDS-staged 256 x 128 tiles: one column tile (N = 128) from 128 rows (W4A16 from 129)
@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("M,K,group", [(130, 2048, 128), (160, 2048, 32), (300, 1024, 256), (257, 512, 64)])
def test_lds_staged(dev, M, K, group, dtype):
    N, cols = 128, (slice(0, 128),)
    _w4a16(dev, M, K, N, group, dtype, _lib.KBH_KERNEL_STAGED, cols)
    _fp8w(dev, M, K, N, group, dtype, _lib.KBH_KERNEL_STAGED, cols)
    if dtype == F16:
        _w8a8(dev, M, K, N, _lib.KBH_KERNEL_STAGED, cols)
        _w8a8(dev, 128, K, N, _lib.KBH_KERNEL_STAGED, cols)


@pytest.mark.parametrize("dtype", [F16, BF16])
def test_lds_staged_no_alloc_and_lora(dev, dtype):
    M, K, N = 160, 2048, 128
    lib = _lib.load()
    assert lib.kbh_w4a16_kernel(M, N, K, 128, DT[dtype], None) == _lib.KBH_KERNEL_STAGED
    d = [t.to(dev) for t in inputs.w4a16(M, K, N, 128, dtype, seed=3)]
    want = ops.w4a16_gemm(*d)
    y = torch.full_like(want, float("nan"))
    st = torch.cuda.current_stream().cuda_stream
    assert lib.kbh_w4a16_gemm_noalloc(*[t.data_ptr() for t in d], y.data_ptr(), M, N, K, 128, DT[dtype], st) == 0
    assert torch.equal(y, want)
    ins = inputs.lora_qgemm(130, 2048, 128, 16, 4, dtype, seed=5)
    out = ops.lora_qgemm(*[t.to(dev) for t in ins])
    cmp = compare(out, ol.forward(*[t.float().numpy() if t.is_floating_point() else t.numpy() for t in ins]))
    assert cmp.ok, cmp


@pytest.mark.parametrize("dtype", [F16, BF16])
def test_lds_staged_dequant_bit_exact(dev, dtype):
    """One-hot x: each output row is a dequantized weight row, rounded once, bit for bit."""
    M, K, N, G = 160, 2048, 128, 128
    dt = "f16" if dtype == F16 else "bf16"
    g = torch.Generator().manual_seed(11)
    ks = torch.randperm(K, generator=g)[:M]
    x = torch.zeros(M, K, dtype=dtype)
    x[torch.arange(M), ks] = 1.0
    q = inputs.random_packed_int4(K, N, g)
    s = (torch.randn(K // G, N, generator=g) * 0.01).to(dtype)
    z = (torch.randint(0, 16, (K // G, N), generator=g).float() + torch.rand(K // G, N, generator=g)).to(dtype)
    y = ops.w4a16_gemm(*[t.to(dev) for t in (x, q, s, z)])
    W = ow.dequant(q.numpy(), s.float().numpy(), z.float().numpy(), dt)
    assert np.array_equal(y.float().cpu().numpy(), W[ks.numpy()])
    codes = torch.randint(0, 256, (K, N), generator=g, dtype=torch.uint8)
    codes[(codes & 0x7F) == 0x7F] = 0x38        # drop the two NaN codes
    s8 = (torch.rand(K // G, N, generator=g) * 4 + 0.01).to(F16)
    y = ops.fp8w_gemm(x.to(dev), codes.view(torch.float8_e4m3fn).to(dev), s8.to(dev))
    W = of.dequant(codes.numpy(), s8.float().numpy(), dt)
    assert np.array_equal(y.float().cpu().numpy(), W[ks.numpy()])


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("M,K,N,group", [(65, 512, 640, 32), (96, 2048, 1408, 128), (128, 1024, 8064, 64), (127, 1024, 384, 256),
                                         (100, 2048, 128, 128)])
def test_128_column_tiles(dev, M, K, N, group, dtype):
    cols = (slice(0, min(N, 256)), slice(N - min(N, 384), N))
    _w4a16(dev, M, K, N, group, dtype, _lib.KBH_KERNEL_NARROW128, cols)
