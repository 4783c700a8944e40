"""The byte-weight GEMM (FP8 weights, and the multi-LoRA base) on the warp-specialised wide tiles,
and K ranges that end in the middle of the kernels' loop iteration.

Edges: row counts about the tile heights of 64 and 128 rows, full and one-row-over tiles, one
column tile, K of an odd number of quantization groups (half an iteration), every block size, and
shapes where the decode kernel's grid exceeds one workgroup per CU (64-row tiles)."""
import numpy as np
import pytest
import torch

from kernelbench_harbor_amd import inputs, ops
from kernelbench_harbor_amd.harness import compare
from oracle import fp8w as of
from oracle import lora as ol
from oracle import w4a16 as ow

pytestmark = pytest.mark.gpu

F16, BF16 = torch.float16, torch.bfloat16
# M, K, N, block
FP8W = [(33, 3584, 3584, 128), (64, 3584, 3584, 64), (65, 768, 256, 256), (128, 896, 256, 128),
        (129, 96 * 4, 512, 32), (256, 320, 256, 64), (257, 1152, 512, 128), (513, 256, 256, 256),
        (300, 128, 256, 32)]


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("M,K,N,block", FP8W)
def test_fp8w_wide(dev, M, K, N, block, dtype):
    print(f"[fp8w wide] M={M} K={K} N={N} B={block} {dtype}", flush=True)
    x, w, s = inputs.fp8w(M, K, N, block, dtype, seed=M + K)
    y = ops.fp8w_gemm(x.to(dev), w.to(dev), s.to(dev))
    cmp = compare(y, of.forward(x.float().numpy(), w.view(torch.uint8).numpy(), s.float().numpy()))
    assert cmp.ok, cmp
    assert torch.equal(y, ops.fp8w_gemm(x.to(dev), w.to(dev), s.to(dev)))


@pytest.mark.parametrize("M,block", [(65, 32), (256, 64), (300, 128), (512, 256)])
@pytest.mark.parametrize("dtype", [F16, BF16])
def test_fp8w_wide_dequant_bit_exact(dev, M, block, dtype):
    """One-hot x: each output row is a dequantized weight row, rounded once, bit for bit."""
    K, N = 1280, 512
    g = torch.Generator().manual_seed(M)
    codes = torch.randint(0, 256, (K, N), generator=g, dtype=torch.int64)
    codes[(codes & 0x7F) == 0x7F] = 0x38        # drop the two NaN codes
    w = codes.to(torch.uint8).view(torch.float8_e4m3fn)
    s = (torch.rand(K // block, N, generator=g) * 4 + 0.01).to(torch.float16)
    ks = torch.randperm(K, generator=g)[:M]
    x = torch.zeros(M, K, dtype=dtype)
    x[torch.arange(M), ks] = 1.0
    y = ops.fp8w_gemm(x.to(dev), w.to(dev), s.to(dev)).float().cpu().numpy()
    W = of.dequant(codes.to(torch.uint8).numpy(), s.float().numpy(), "f16" if dtype == F16 else "bf16")
    assert np.array_equal(y, W[ks.numpy()])


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("T", [65, 129, 257])
def test_lora_wide_base_matches_native_rounding(dev, T, dtype):
    """One-hot activations and dyadic adapters (every sum exact in fp32), any int8 value in the
    base weight: bit-exact against the oracle's native path on 128-row tiles (N = 256 is one column tile,
    so the estimate never picks 256 rows)."""
    D, N, r, L = 640, 256, 16, 3
    g = torch.Generator().manual_seed(T)
    q = torch.randint(-128, 128, (D, N), generator=g, dtype=torch.int8)
    s = (torch.rand(D // 128, N, generator=g) * 0.1).to(dtype)
    A = (torch.randint(-8, 8, (L, D, r), generator=g).float() / 16).to(dtype)
    B = (torch.randint(-8, 8, (L, r, N), generator=g).float() / 64).to(dtype)
    ids = torch.randint(0, L, (T,), generator=g)
    x = torch.zeros(T, D, dtype=dtype)
    x[torch.arange(T), torch.randint(0, D, (T,), generator=g)] = 1.0
    y = ops.lora_qgemm(*[t.to(dev) for t in (x, q, s, A, B, ids)]).float().cpu().numpy()
    ins = [t.float().numpy() if t.is_floating_point() else t.numpy() for t in (x, q, s, A, B, ids)]
    want = ol.forward(*ins, dtype="f16" if dtype == F16 else "bf16")
    assert np.array_equal(y, want), np.abs(y - want).max()


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("M,K,N,group", [(33, 384, 256, 128), (64, 2304, 512, 256), (65, 640, 256, 128),
                                         (128, 192, 256, 64), (257, 896, 512, 128), (300, 768, 256, 256)])
def test_w4a16_odd_number_of_groups(dev, M, K, N, group, dtype):
    """K of an odd number of half iterations: the wide kernels leave their loop in its middle."""
    x, q, s, z = inputs.w4a16(M, K, N, group, dtype, seed=M)
    y = ops.w4a16_gemm(*[t.to(dev) for t in (x, q, s, z)])
    cmp = compare(y, ow.forward(x.float().numpy(), q.numpy(), s.float().numpy(), z.float().numpy()))
    assert cmp.ok, cmp


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("M,K,group", [(2100, 256, 256), (2100, 640, 128), (8200, 128, 128)])
def test_w4a16_half_iteration_tails(dev, M, K, group, dtype):
    """K ranges that end (or lie wholly) in half an iteration, on many workgroups at once: there
    the compiler drops the raw-word loads past the end, so the wait for the staged x rows may count
    the x loads alone. Every row against the oracle, and twice the same bits."""
    N = 256
    x, q, s, z = inputs.w4a16(M, K, N, group, dtype, seed=M)
    d = [t.to(dev) for t in (x, q, s, z)]
    y = ops.w4a16_gemm(*d)
    gt = torch.from_numpy(np.asarray(ow.forward(x.float().numpy(), q.numpy(), s.float().numpy(),
                                                z.float().numpy())))
    err = (y.float().cpu() - gt).abs().amax(dim=1) / gt.abs().amax()
    # one rounding of the output and one of each weight: 2^-8 (bf16) covers both in every row
    assert err.max() <= 2.0 ** -8, (int(err.argmax()), float(err.max()))
    for _ in range(3):
        assert torch.equal(y, ops.w4a16_gemm(*d))


# M, K, N: a last column tile that overlaps its neighbour (N % 256 == 128), K ranges of uneven
# length (units that no split count near the 256 workgroups divides). The plans are 64- and 128-row
# tiles and, where that is faster, the decode kernel; the 256-row tiles' edges are in test_gpu_routes.py.
WIDE_EDGES = [(33, 1152, 384), (129, 2176, 384), (200, 18944, 640), (300, 1408, 896), (257, 128, 384),
              (64, 9472, 1152), (17, 18944, 2176), (32, 9472, 4224)]  # 17-32 rows: 64/128-row tiles


@pytest.mark.parametrize("M,K,N", WIDE_EDGES)
def test_w8a8_wide_edges_bit_exact(dev, M, K, N):
    g = torch.Generator().manual_seed(M + K)
    x = torch.randint(-128, 128, (M, K), generator=g, dtype=torch.int8)
    w = torch.randint(-128, 128, (K, N), generator=g, dtype=torch.int8)
    acc = ops.w8a8_gemm_i32(x.to(dev), w.to(dev)).cpu().numpy()
    # exact: |sum| <= K * 2^14 < 2^53
    want = x.double().numpy() @ w.double().numpy()
    assert np.array_equal(acc.astype(np.float64), want)


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("M,K,N", WIDE_EDGES)
def test_wide_edges_match_oracle(dev, M, K, N, dtype):
    x, q, s, z = inputs.w4a16(M, K, N, 128, dtype, seed=M)
    y = ops.w4a16_gemm(*[t.to(dev) for t in (x, q, s, z)])
    cmp = compare(y, ow.forward(x.float().numpy(), q.numpy(), s.float().numpy(), z.float().numpy()))
    assert cmp.ok, cmp
    x, w, s = inputs.fp8w(M, K, N, 128, dtype, seed=M)
    y = ops.fp8w_gemm(x.to(dev), w.to(dev), s.to(dev))
    cmp = compare(y, of.forward(x.float().numpy(), w.view(torch.uint8).numpy(), s.float().numpy()))
    assert cmp.ok, cmp


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("T,D,N,r,L", [(1, 128, 128, 4, 1), (5, 4096, 384, 64, 3), (16, 1056, 256, 32, 2),
                                       (32, 2048, 512, 8, 4), (33, 4096, 4096, 16, 8)])
def test_lora_shrink_beside_decode(dev, T, D, N, r, L, dtype):
    """The shrink as further workgroups of the base GEMM's launch (up to 32 rows: one and two row
    blocks, fewer waves than four, D ranges shorter than a step) and as its own launch (33)."""
    x, q, s, A, B, ids = inputs.lora_qgemm(T, D, N, r, L, dtype, seed=T + D)
    if D % 128:
        s = (torch.randn(D // 32, N, generator=torch.Generator().manual_seed(1)) * 0.01).to(dtype)
    ins = [x, q, s, A, B, ids]
    y = ops.lora_qgemm(*[t.to(dev) for t in ins])
    cmp = compare(y, ol.forward(*[t.float().numpy() if t.is_floating_point() else t.numpy() for t in ins]))
    assert cmp.ok, cmp
    assert torch.equal(y, ops.lora_qgemm(*[t.to(dev) for t in ins]))
