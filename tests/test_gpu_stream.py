"""The streaming kernels (up to 16 rows per tile): W4A16 (the SiLU FFN at decode batches, dense rows)
and FP8 weights, against the float64 oracle. Edges: one token, an expert of exactly 16 and of 17 rows (a second tile), experts
without rows, K ranges with fewer units than waves and uneven over waves and splits, every group
size."""
import numpy as np
import pytest
import torch

from kernelbench_harbor_amd import _lib, inputs, ops
from kernelbench_harbor_amd.harness import compare
from oracle import fp8w as of
from oracle import qmoe as oq
from oracle import w4a16 as ow

pytestmark = pytest.mark.gpu

F16, BF16 = torch.float16, torch.bfloat16


def _np(ins):
    return [t.float().numpy() if t.is_floating_point() else t.numpy() for t in ins]


def _logits(counts, seed):
    """fp32 logits whose top-2 give expert e exactly counts[e] of the 2T slots (no count above T)."""
    L = np.repeat(np.arange(len(counts)), counts)
    T = len(L) // 2
    rng = np.random.default_rng(seed)
    lg = rng.normal(size=(T, len(counts))).astype(np.float32) - 4.0
    lg[np.arange(T), L[:T]] = 3.0 + rng.uniform(0, 1, T)
    lg[np.arange(T), L[T:]] = 1.0 + rng.uniform(0, 1, T)
    return torch.from_numpy(lg)


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("counts,D,F,group", [
    ([1, 1, 0, 0], 256, 512, 128),             # one token; 2 units of K for 4 waves
    ([16, 17, 1, 0, 14], 768, 512, 128),       # 16 and 17 rows; 6 units
    ([33, 20, 13, 0], 512, 1280, 64),          # three tiles of one expert; 20 uneven units
    ([5, 3, 9, 7], 1792, 256, 256),            # 7 units of 256 rows
    ([12, 20, 2, 14], 1280, 768, 32),
])
def test_ffn_stream(dev, counts, D, F, group, dtype):
    T, E = sum(counts) // 2, len(counts)
    print(f"[ffn stream] {counts} D={D} F={F} g{group} {dtype}", flush=True)
    ins = inputs.qmoe_ffn(T, D, F, E, group=group, dtype=dtype, seed=D + F)
    ins[1] = _logits(counts, D)
    topi, _ = oq.route_top2(ins[1].numpy())
    assert np.bincount(topi.ravel(), minlength=E).tolist() == counts
    y = ops.qmoe_ffn(*[t.to(dev) for t in ins])
    cmp = compare(y, oq.ffn_forward(*_np(ins)))
    assert cmp.ok, cmp
    ops.scratches.get(0, dev).fill_(255)   # no content requirement on the workspace
    assert torch.equal(y, ops.qmoe_ffn(*[t.to(dev) for t in ins]))


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("group", [32, 128])
def test_ffn_stream_non_finite(dev, dtype, group):
    """Infinities and NaN in x, and a column of h that leaves the type's range: the streamed rows agree
    with the same tokens in a batch on the wide tiles, sign by sign (an infinity in one column of h meets each
    down weight's sign), and the other rows are the same bits as without the values in x."""
    E, D, F, T = 4, 512, 768, 20
    ins = inputs.qmoe_ffn(64, D, F, E, group=group, dtype=dtype, seed=9)
    ins[6][:, :, 100] *= 2.0 ** 17           # up scales: h[:, 100] is past 65504 in many rows
    clean = [t.to(dev) for t in ins]
    x = ins[0].clone()
    big = torch.finfo(dtype).max
    x[1, 17] = float("inf")
    x[3, 5], x[3, 300] = float("inf"), float("-inf")
    x[4, 100] = float("nan")
    x[6, :] = x[6, :] * (1.5 if dtype == F16 else 2e18)      # bf16: past 3.4e38 in that column alone
    x[9, :] = x[9, :] * (1.5 if dtype == F16 else 2e18)
    x[7, 200] = -big
    x[8, 40], x[8, 41] = 0.9 * big, 0.9 * big
    x[13, D - 1] = float("-inf")
    dirty = [x.to(dev)] + clean[1:]
    few = lambda d: [d[0][:T].contiguous(), d[1][:T].contiguous(), *d[2:]]
    assert 2 * T < 32 * E <= 2 * 64    # streamed, and on the wide tiles
    got, want = ops.qmoe_ffn(*few(dirty)).float(), ops.qmoe_ffn(*dirty)[:T].float()
    assert torch.isnan(want).any() and torch.isinf(want).any()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    inf = torch.isinf(want)
    assert torch.equal(torch.isinf(got), inf) and torch.equal(got[inf], want[inf])
    fin = torch.isfinite(want)
    # The wide tiles' weights are rounded to the type (2^-11 / 2^-8 of each, so of a column's sum of typical
    # size, not of a sum that cancels), and h and o once on both sides: 2^-8 / 2^-5 of the largest output
    # of the rows of natural size, or of the row.
    eps = 2.0 ** -8 if dtype == F16 else 2.0 ** -5
    scale = torch.where(fin, want, 0).abs().amax(dim=1, keepdim=True)
    natural = [r for r in range(T) if r not in (6, 9)]
    scale = torch.maximum(scale, scale[natural].max())
    assert ((got - want).abs()[fin] <= (eps * scale.expand_as(want))[fin]).all()
    touched = torch.tensor([1, 3, 4, 6, 7, 8, 9, 13])
    same = torch.ones(T, dtype=torch.bool)
    same[touched] = False
    assert torch.equal(got.cpu()[same].nan_to_num(), ops.qmoe_ffn(*few(clean)).float().cpu()[same].nan_to_num())


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("D,F", [(256, 5376), (8448, 256)])
def test_ffn_stream_passes(dev, D, F, dtype):
    """Slices past 64 MiB: two passes over the columns (11 and 10 tiles of gate/up, 17 and 16 of down)."""
    T, E = 1000, 64
    ins = inputs.qmoe_ffn(T, D, F, E, group=128, dtype=dtype, seed=2)
    assert 2 * T * (2 * F if F > D else D) * 4 > 64 << 20
    d = [t.to(dev) for t in ins]
    y = ops.qmoe_ffn(*d)
    a = _np(ins)
    rows = np.r_[0:24, T - 24:T]
    cmp = compare(y[torch.from_numpy(rows).to(dev)], oq.ffn_forward(a[0][rows], a[1][rows], *a[2:]))
    assert cmp.ok, cmp
    ops.scratches.get(0, dev).fill_(255)   # no content requirement on the workspace
    assert torch.equal(y, ops.qmoe_ffn(*d))


def test_ffn_stream_full_width(dev):
    """The benchmark's layer (D=4096, F=14336, E=8) at 9 tokens, the last 256 output columns."""
    ins = inputs.qmoe_ffn(T=9, seed=5)
    y = ops.qmoe_ffn(*[t.to(dev) for t in ins]).float().cpu().numpy()
    a = _np(ins)
    down = [a[8][:, :, -32:], a[9][:, :, -256:], a[10][:, :, -256:]]
    cmp = compare(y[:, -256:], oq.ffn_forward(*a[:8], *down))
    assert cmp.ok, cmp


# K, N, group, K splits at M = 16: shapes whose decode grid is several workgroups per CU
DENSE = [(18944, 2048, 128, 32), (18944, 2048, 64, 32), (9472, 4096, 32, 16), (4864, 8448, 256, 4),
         (2048, 66304, 64, 2)]


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("M", [1, 16, 17, 32])
@pytest.mark.parametrize("K,N,group,splits", DENSE)
def test_w4a16_stream(dev, K, N, group, splits, M, dtype):
    """Dense rows: whole and partial 16-row tiles, uneven K ranges, unsplit K (M > 17 of the last shape); the first and last
    256 columns against the oracle, and the no-alloc entry point's bits."""
    if M == 16:  # the streaming plan (its slices)
        assert _lib.load().kbh_w4a16_workspace_bytes(M, N, K, group) == splits * M * N * 4
    x, q, s, z = inputs.w4a16(M, K, N, group, dtype, seed=M + K)
    d = [t.to(dev) for t in (x, q, s, z)]
    y = ops.w4a16_gemm(*d)
    for c in (slice(0, 256), slice(N - 256, N)):
        w = slice(c.start // 8, c.stop // 8)
        gt = ow.forward(x.float().numpy(), q[:, w].numpy(), s[:, c].float().numpy(), z[:, c].float().numpy())
        cmp = compare(y[:, c], gt)
        assert cmp.ok, cmp
    y2 = torch.empty_like(y)
    code = 0 if dtype == F16 else 1
    st = torch.cuda.current_stream().cuda_stream
    assert _lib.load().kbh_w4a16_gemm_noalloc(*[t.data_ptr() for t in d], y2.data_ptr(), M, N, K,
                                              group, code, st) == 0
    assert torch.equal(y, y2)


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("T,D,N,E,group", [(1, 2048, 128, 60, 128), (3, 768, 256, 200, 256), (9, 1280, 128, 65, 64),
                                           (2, 256, 128, 4, 32), (5, 4096, 384, 129, 128)])
def test_qmoe_split_k(dev, T, D, N, E, group, dtype):
    """The reference qMoE op at small batches (K split over workgroups, slices summed by the
    combine) and route tables of one to four waves of experts."""
    ins = inputs.qmoe(T, D, E, N, dtype, seed=T + E, group=group)
    y = ops.qmoe(*[t.to(dev) for t in ins])
    cmp = compare(y, oq.qmoe_forward(*_np(ins)))
    assert cmp.ok, cmp
    ops.scratches.get(0, dev).fill_(255)
    assert torch.equal(y, ops.qmoe(*[t.to(dev) for t in ins]))


# K, N, block: layers whose decode grid is over 512 workgroups. Uneven chunks over splits and waves,
# unsplit K, an odd chunk count, fewer chunks than waves.
FP8W = [(3584, 18944, 128), (9472, 7168, 32), (320, 65664, 64), (192, 65664, 32), (2304, 31872, 256)]


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("M", [1, 7, 16])
@pytest.mark.parametrize("K,N,block", FP8W)
def test_fp8w_stream(dev, K, N, block, M, dtype):
    print(f"[fp8w stream] M={M} K={K} N={N} B={block} {dtype}", flush=True)
    x, w, s = inputs.fp8w(M, K, N, block, dtype, seed=M + K)
    d = [t.to(dev) for t in (x, w, s)]
    y = ops.fp8w_gemm(*d)
    codes = w.view(torch.uint8).numpy()
    for c in (slice(0, 128), slice(N - 128, N)):
        cmp = compare(y[:, c], of.forward(x.float().numpy(), codes[:, c], s[:, c].float().numpy()))
        assert cmp.ok, cmp
    ops.workspaces.get(0, dev).fill_(255)   # no content requirement on the workspace
    assert torch.equal(y, ops.fp8w_gemm(*d))


@pytest.mark.parametrize("dtype", [F16, BF16])
def test_fp8w_stream_dequant_bit_exact(dev, dtype):
    """One-hot x: each output row is a dequantized weight row, rounded once, bit for bit."""
    K, N, block = 2304, 31872, 128
    g = torch.Generator().manual_seed(3)
    codes = torch.randint(0, 256, (K, N), generator=g, dtype=torch.uint8)
    codes[(codes & 0x7F) == 0x7F] = 0x38        # drop the two NaN codes
    s = (torch.rand(K // block, N, generator=g) * 4 + 0.01).to(torch.float16)
    ks = torch.randperm(K, generator=g)[:16]
    x = torch.zeros(16, K, dtype=dtype)
    x[torch.arange(16), ks] = 1.0
    y = ops.fp8w_gemm(x.to(dev), codes.view(torch.float8_e4m3fn).to(dev), s.to(dev))
    W = of.dequant(codes[ks].numpy(), s[ks // block].float().numpy(), "f16" if dtype == F16 else "bf16")
    assert np.array_equal(y.float().cpu().numpy(), W)
