// W4A16 packed-asymmetric group-quantized GEMM for gfx950.
//
// Semantics (reference tasks/quant_w4a16_pa/*/environment/reference.py:10-17):
//   w[k, n] = (((qweight[k, n/8] >> 4*(n%8)) & 0xF) - zeros[k/G, n]) * scales[k/G, n]
//   y       = x @ w
//
// Two kernels:
//
// w4a16_decode_kernel (M <= 16 per 16-row block; HBM-bound decode shapes)
//  * A wavefront owns 128*NW output columns and SPW consecutive 32-row K steps; every load of
//    the wavefront (SPW*8 rows of NW packed words per lane, plus its x fragments) is issued
//    before any arithmetic so that the whole chip's weight stream is in flight at once.
//    Lane l reads qweight[k0 + 8(l/16) + i][n0/8 + (l%16)*NW + w], i = 0..7.
//  * Nibbles become fp16/bf16 MFMA B-fragments with no per-weight arithmetic: one v_perm_b32
//    places byte j of the words of rows k, k+1 into the two 16-bit halves and one v_and_or_b32
//    with a magic exponent turns nibble q into the value B+q (fp16: 1024+q, or 1024+16q for the
//    high nibble; bf16: 128+q). Each (word, nibble) pair feeds one 16x16x32 MFMA whose 16 output
//    columns lie 8*NW apart in n.
//  * Zero points and scales are applied once per quantization group on the fp32 accumulators:
//      sum_k x_k (q_k - z) s = s * (sum_k x_k (B + f q_k) / f - (B/f + z) * sum_k x_k)
//    with sum_k x_k from one extra MFMA against a ones fragment.
//  * The waves of a workgroup (consecutive K ranges of one column tile) reduce through private
//    LDS slices; each workgroup (K split) stores its tile into its own workspace slice, and
//    splitk_sum_kernel, run on the XCDs that wrote them, adds the slices in split order and
//    converts to the output dtype (splitk.h). Workgroup ids are remapped so that all K splits
//    of a column tile run on one XCD.
//
// Larger M (M > 32, except where the decode kernel stays faster): tiled_wide_gemm (tiled_wide.h) with
// W4WidePolicy, which dequantizes each packed 32 x TN weight slab once per workgroup into LDS with the exact reference arithmetic
// ((q - z) rounded to the input dtype, times s rounded), in MFMA fragment order; x goes from
// global memory straight into MFMA registers. Split-K partial sums use the caller's scratch.
// Shapes it does not cover fall back to tiled_f16_gemm (256 x 128 LDS-staged tiles) or to the
// decode kernel.
#include "kbh_common.h"
#include "splitk.h"
#include "tiled_f16.h"
#include "tiled_wide.h"
#include "tiled_ws.h"
#include "tiled_ws256.h"
#include "w4_dequant.h"
#include "w4_stream.h"

namespace kbh {
namespace {

// ======================================================================================
// Decode kernel
// ======================================================================================

// SPG = K steps per quantization group when a group is shorter than a wave's K range
// (SPG < SPW), otherwise SPG == SPW (each wave lies inside one group). The fold schedule is thus
// static, and the scales/zeros of every group a wave touches are loaded with its weights.
template <int NW, int SPW, int SPG, bool BF16>
__global__ __launch_bounds__(kSplitKMaxWaves * 64) void w4a16_decode_kernel(
    const uint16_t* __restrict__ x, const uint32_t* __restrict__ qw,
    const uint16_t* __restrict__ scales, const uint16_t* __restrict__ zeros,
    uint16_t* __restrict__ y, float* __restrict__ acc, int M, int N, int K, int group,
    int splits) {
  constexpr int NWG = 128 * NW;  // output columns of one workgroup
  constexpr int NCS = 8 * NW;    // MFMA column sets per wave
  constexpr uint32_t MAGIC = BF16 ? kMagicBF16 : kMagicF16;
  __shared__ SplitKSmem<NCS, float> sm;

  const int waves = blockDim.x >> 6;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: SGPR addressing
  const int c = lane & 15;
  const int g = lane >> 4;
  const int id = xcd_remap(blockIdx.x, gridDim.x);
  const int tile = id / splits;
  const int split = id - tile * splits;
  const int n0 = tile * NWG;
  const int m0 = blockIdx.y * 16;
  const int st0 = (split * waves + wave) * SPW;  // first 32-row K step of this wave
  const int NP = N >> 3;

  // ---- every load of this wave, up front ----------------------------------------------
  // x fragments and group constants first: loads complete in issue order, so the MFMAs of
  // step u can start as soon as step u's weights arrive, while later steps are still in flight.
  kbh_u32x4 af[SPW];
  const bool xok = m0 + c < M;
  const uint16_t* xb = x + (size_t)(xok ? m0 + c : 0) * K + st0 * 32 + 8 * g;
#pragma unroll
  for (int u = 0; u < SPW; ++u) af[u] = *reinterpret_cast<const kbh_u32x4*>(xb + u * 32);
  constexpr int NG = SPW / SPG;  // quantization groups touched by this wave
  kbh_u32x4 sv[NG][NW], zv[NG][NW];
#pragma unroll
  for (int gq = 0; gq < NG; ++gq) {
    const int gi = ((st0 + gq * SPG) << 5) / group;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const size_t off = (size_t)gi * N + n0 + 8 * (c * NW + w);
      sv[gq][w] = *reinterpret_cast<const kbh_u32x4*>(scales + off);
      zv[gq][w] = *reinterpret_cast<const kbh_u32x4*>(zeros + off);
    }
  }
  __builtin_amdgcn_sched_barrier(0);  // keeps the group constants ahead of the weight stream
  uint32_t wd[SPW][8][NW];
  // Buffer loads from the wave's first row: the row offset is an SGPR (soffset) and the lane
  // offset one VGPR, so no load needs per-lane 64-bit address arithmetic (global loads got a
  // v_lshl_add_u64 chain). Reads past the matrix would return zero (range-checked resource).
  const size_t qbase = (size_t)st0 * 32 * NP + (n0 >> 3);
  const __amdgpu_buffer_rsrc_t qres = make_rsrc(qw + qbase, ((size_t)K * NP - qbase) * 4);
  const uint32_t qlane = (uint32_t)(8 * g * NP + c * NW) * 4u;
#pragma unroll
  for (int u = 0; u < SPW; ++u) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int soff = (u * 32 + i) * NP * 4;
      if constexpr (NW == 2) {
        const kbh_u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(qres, qlane, soff, kBufNT);
        wd[u][i][0] = v[0];
        wd[u][i][1] = v[1];
      } else {
        wd[u][i][0] = __builtin_amdgcn_raw_buffer_load_b32(qres, qlane, soff, kBufNT);
      }
    }
  }
  // Nothing may use a loaded value before the last load is issued: a consumer scheduled between
  // the loads makes the wave wait one memory latency with part of its stream not yet requested.
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < SPW; ++u)
    if (!xok) af[u] = kbh_u32x4{0u, 0u, 0u, 0u};  // rows past M contribute zero

  const uint32_t one = BF16 ? kOneBF16 : kOneF16;
  const kbh_u32x4 ones = {one, one, one, one};
  // The nibble masks in SGPRs and the magic exponent in a VGPR: (P & mask) | magic is then one
  // v_and_or_b32 (a VOP3 here takes no literal and reads at most one SGPR); with literals the
  // compiler emits a v_and_b32 and a v_or_b32 per B dword.
  uint32_t mlo = 0x000F000Fu, mhi = 0x00F000F0u, magic = MAGIC;
  asm volatile("" : "+s"(mlo), "+s"(mhi));
  asm volatile("" : "+v"(magic));
  kbh_f32x4 tot[NCS], part[NCS], xs = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int cs = 0; cs < NCS; ++cs) {
    tot[cs] = kbh_f32x4{0.f, 0.f, 0.f, 0.f};
    part[cs] = tot[cs];
  }
#pragma unroll
  for (int u = 0; u < SPW; ++u) {
    xs = mfma16x16x32<BF16>(af[u], ones, xs);
#pragma unroll
    for (int w = 0; w < NW; ++w) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        kbh_u32x4 blo, bhi;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          const uint32_t P = pair_bytes_rt(wd[u][2 * p][w], wd[u][2 * p + 1][w], j);
          blo[p] = (P & mlo) | magic;
          bhi[p] = BF16 ? (((P >> 4) & mlo) | magic) : ((P & mhi) | magic);
        }
        part[w * 8 + 2 * j] = mfma16x16x32<BF16>(af[u], blo, part[w * 8 + 2 * j]);
        part[w * 8 + 2 * j + 1] = mfma16x16x32<BF16>(af[u], bhi, part[w * 8 + 2 * j + 1]);
      }
    }
    // Fold at the end of each quantization group (static schedule).
    if ((u + 1) % SPG == 0) {
      const int gq = u / SPG;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
#pragma unroll
        for (int nib = 0; nib < 8; ++nib) {
          const uint32_t sw = sv[gq][w][nib >> 1], zw = zv[gq][w][nib >> 1];
          const uint16_t sh = (uint16_t)((nib & 1) ? (sw >> 16) : (sw & 0xffffu));
          const uint16_t zh = (uint16_t)((nib & 1) ? (zw >> 16) : (zw & 0xffffu));
          const float s = half_bits_to_f32<BF16>(sh);
          const float z = half_bits_to_f32<BF16>(zh);
          const float a = (!BF16 && (nib & 1)) ? 0.0625f : 1.0f;
          const float bz = (BF16 ? 128.0f : ((nib & 1) ? 64.0f : 1024.0f)) + z;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float t = fmaf(-bz, xs[i], part[w * 8 + nib][i] * a);
            tot[w * 8 + nib][i] = fmaf(s, t, tot[w * 8 + nib][i]);
          }
          part[w * 8 + nib] = kbh_f32x4{0.f, 0.f, 0.f, 0.f};
        }
      }
      xs = kbh_f32x4{0.f, 0.f, 0.f, 0.f};
    }
  }

  // The fold's only use is inside splitk_reduce's row-guarded branch; without this the compiler
  // sinks the fold, and the group-constant loads with it, behind that branch and the last weight.
#pragma unroll
  for (int cs = 0; cs < NCS; ++cs) asm volatile("" : "+v"(tot[cs]));
  const int rows = min(16, M - m0);
  splitk_reduce<NCS, float>(tot, sm, acc, split, splits, rows, M, N, m0, n0, [&](int r, int n, float v) {
    y[(size_t)(m0 + r) * N + n0 + n] = f32_to_half_bits<BF16>(v);
  });
}

constexpr int kWideMinM = 33;  // rows from which the wide tiles take over (below)

struct DecodePlan {
  int nw, spw, spg, waves, ntiles, splits, mblocks;
};

// The (NW, SPW, SPG) instantiations of w4a16_decode_kernel; plan_decode picks only from these.
// NW = 2 takes at most two quantization groups per wave (SPW / SPG <= 2): more groups' constants
// on top of 256 columns' accumulators spill. SPW = 8 exists only with NW = 2 (NW = 1 was measured
// slower with it on every shape swept).
#define KBH_DECODE_VARIANTS(X)                                                                   \
  X(2, 8, 8) X(2, 8, 4) X(2, 4, 4) X(2, 4, 2) X(2, 2, 2) X(2, 2, 1) X(2, 1, 1) X(1, 4, 4)         \
  X(1, 4, 2) X(1, 4, 1) X(1, 2, 2) X(1, 2, 1) X(1, 1, 1)

bool decode_variant_built(int nw, int spw, int spg) {
#define KBH_DEC_IS(NW_, SPW_, SPG_) if (nw == NW_ && spw == SPW_ && spg == SPG_) return true;
  KBH_DECODE_VARIANTS(KBH_DEC_IS)
#undef KBH_DEC_IS
  return false;
}

// Estimated duration (µs, up to a constant) of a decode launch plus its split-K sum. Every load
// of a workgroup is in flight at once, so a CU's time is set by the weight bytes of the
// workgroups it runs one after another (KB = 2 per K step per 128 columns) plus a fixed cost per
// workgroup (halved when two fit on a CU: NW = 1 needs half the LDS), and fewer waves issue
// those bytes more slowly; the split-K slices add a write and a read of splits x M x N fp32.
// The constants are a least-squares fit to a sweep of every (NW, SPW, waves) plan on MI355X
// over the shapes K x N = 4096 x 14336, 14336 x 4096, 8192 x 28672, 28672 x 8192,
// 3584 x 18944, 18944 x 3584, 8192 x 29568 and 29568 x 8192 at M = 1 and 16 (group 128): the
// plan it picks is within 2% of the sweep's fastest NW = 2 plan on all 16, where the former
// "grid closest to one workgroup per CU" rule lost up to 28%.
float decode_cost(int M, int N, int nw, int spw, int waves, int splits, int grid) {
  const float kb = 2.0f * spw * waves * nw;
  const float slowdown = 1.0f + 0.53f * (8 - waves) / 8.0f;
  const int per_cu = (grid + 255) / 256;
  float t = per_cu * ((nw == 1 ? 0.9f : 1.8f) + kb * slowdown / 23.3f);
  if (splits > 1) t += (float)splits * M * N * 8.0f / 1024.0f / 2540.0f;
  return t;
}

// Chooses column width (NW: 128*NW columns per workgroup), K steps per wave (SPW) and waves per
// workgroup (the K steps divide evenly) by decode_cost. NW = 2 whenever N allows it (NW = 1 plans
// that the cost prefers there were measured slower on most shapes: half-width rows per load),
// except with 32-row groups, where NW = 2 holds at most SPW = 2 and NW = 1 with SPW = 4
// measured 4-11% faster.
bool plan_decode(int M, int N, int K, int group_steps_, DecodePlan* p) {
  const int nsteps = K / 32;
  const int gsteps = group_steps_;  // 1, 2, 4 or 8 (group 32..256); divides nsteps
  const int nw = (N % 256 == 0 && gsteps > 1) ? 2 : 1;
  const int ntiles = N / (128 * nw);
  const int mblocks = (M + 15) / 16;
  float best = 0.0f;
  p->waves = 0;
  for (int spw = 8; spw >= 1; spw >>= 1) {
    if (nsteps % spw != 0) continue;
    // Wave ranges start at multiples of SPW steps, so they stay inside one group when the group
    // spans a multiple of SPW steps; otherwise the group (1, 2 or 4 steps) divides SPW.
    const int spg = (gsteps % spw == 0) ? spw : gsteps;
    if (!decode_variant_built(nw, spw, spg)) continue;
    const int units = nsteps / spw;
    for (int w = kSplitKMaxWaves; w >= 1; --w) {
      if (units % w != 0) continue;
      const int splits = units / w;
      const float c = decode_cost(M, N, nw, spw, w, splits, ntiles * splits * mblocks);
      if (p->waves == 0 || c < best) {
        best = c;
        *p = DecodePlan{nw, spw, spg, w, ntiles, splits, mblocks};
      }
    }
  }
  return p->waves > 0;
}

template <int NW, int SPW, int SPG, bool BF16>
void launch_decode(const DecodePlan& p, const void* x, const int32_t* qw, const void* s,
                   const void* z, void* y, float* acc, int M, int N, int K, int group,
                   hipStream_t stream) {
  dim3 grid(p.ntiles * p.splits, p.mblocks);
  hipLaunchKernelGGL((w4a16_decode_kernel<NW, SPW, SPG, BF16>), grid, dim3(p.waves * 64), 0, stream,
                     (const uint16_t*)x, (const uint32_t*)qw, (const uint16_t*)s,
                     (const uint16_t*)z, (uint16_t*)y, acc, M, N, K, group, p.splits);
  if (p.splits > 1)
    launch_splitk_sum(reinterpret_cast<const kbh_f32x4*>(acc), HalfOut<BF16>{(uint16_t*)y, N}, M, N,
                      p.ntiles, 128 * NW, p.splits, stream);
}

// The streaming kernel (w4_stream.h) takes the calls that the decode kernel runs in several rounds
// of workgroups, each of which fills and drains the memory pipeline: large layers, two row blocks,
// and K x N that no wave split divides well (K = 11008, 18944, 29568). The two estimates
// decide. Measured (decode -> stream, us, group 128 fp16) at M=16: 11008 x 4096 19.8 -> 13.7,
// 18944 x 3584 23.9 -> 16.6, 28672 x 8192 38.9 -> 32.8, 29568 x 8192 51.3 -> 34.1, 8192 x 28672
// 37.6 -> 35.8, 4096 x 128256 74.1 -> 56.9; M=32: 36.4 -> 16.0, 38.1 -> 23.5, 71.4 -> 49.3, 90.5 ->
// 51.5, 70.2 -> 58.0, 140 -> 115. One-round grids stay with the decode kernel (14336 x 4096 M=16
// 13.1 against 14.4, 4096 x 14336 13.1 / 14.7), as does an unsplit K (it writes y itself: K=512
// N=66304 M=16 11.6 / 14.9). Returns the K splits, 0 for the decode kernel.
int plan_stream(const DecodePlan& d, int M, int N, int K, int group) {
  if (M >= kWideMinM || d.splits == 1 || !w4_stream_ok(N, K, group)) return 0;
  const int mb = (M + 15) / 16;
  const int s = w4_stream_splits(M, N, K, group, mb, 1);
  // Where either plan's slices exceed the no-alloc entry point's array (they are written also when
  // K is unsplit), the decode plan stays: that entry point accepts and refuses what it always has.
  if ((size_t)s * M * N * 4 > KBH_W4A16_NOALLOC_SCRATCH_BYTES ||
      splitk_workspace_bytes(M, N, d.splits) > KBH_W4A16_NOALLOC_SCRATCH_BYTES)
    return 0;
  const float dec = decode_cost(M, N, d.nw, d.spw, d.waves, d.splits, d.ntiles * d.splits * d.mblocks);
  return w4_stream_cost(M, N, K, mb, 1, s) < dec ? s : 0;
}

// Workspace of a call on the decode or the streaming kernel.
size_t decode_workspace_bytes(const DecodePlan& d, int M, int N, int K, int group) {
  const int s = plan_stream(d, M, N, K, group);
  return s > 0 ? round_up((size_t)s * M * N * 4, 256) : splitk_workspace_bytes(M, N, d.splits);
}

template <bool BF16>
void launch_dense_stream(int splits, const void* x, const int32_t* qw, const void* s, const void* z,
                         void* y, float* slices, int M, int N, int K, int group, hipStream_t st) {
  W4StreamArgs a{};
  a.x = (const uint16_t*)x;
  a.mat[0] = a.mat[1] = W4Mat{(const uint32_t*)qw, (const uint16_t*)s, (const uint16_t*)z};
  a.slices = slices;
  a.M = M;
  a.ld = a.N = N;
  a.K = K;
  a.group = group;
  a.splits = splits;
  a.tiles0 = N / kStreamCols;
  launch_w4_stream<BF16, false>(a, a.tiles0, (M + 15) / 16, st);
  launch_splitk_sum(reinterpret_cast<const kbh_f32x4*>(slices), HalfOut<BF16>{(uint16_t*)y, N}, M,
                    N, a.tiles0, kStreamCols, splits, st);
}

template <bool BF16>
void dispatch_decode(const DecodePlan& p, const void* x, const int32_t* qw, const void* s,
                     const void* z, void* y, float* acc, int M, int N, int K, int group,
                     hipStream_t st) {
#define KBH_DEC(NW_, SPW_, SPG_)                                                                 \
  if (p.nw == NW_ && p.spw == SPW_ && p.spg == SPG_)                                             \
    return launch_decode<NW_, SPW_, SPG_, BF16>(p, x, qw, s, z, y, acc, M, N, K, group, st);
  KBH_DECODE_VARIANTS(KBH_DEC)
#undef KBH_DEC
}

// ======================================================================================
// Large-M kernels
// ======================================================================================
// Above kWideMinM rows the wide-tile kernel (tiled_wide.h) takes over from the split-K decode
// kernel: up to 64 rows, 64 x 256 tiles; up to 128 rows, 128 x 256 tiles with one workgroup per
// CU (128 x 128 tiles, two per CU, when N is 128); above, 128 x 256 or 256 x 256 tiles by the
// planner's estimate (plan_wide). The 256-column tiles run
// with a 4-slab prefetch ring; those of 64 and 128 rows on the warp-specialised kernel
// (tiled_ws.h: 4 dequantizing and 4 MFMA waves per workgroup), those of 256 rows on its 12-wave
// form (tiled_ws256.h: 4 waves stage weights and x, 8 MFMA waves; K=14336 N=4096 M=1024
// 153.0 -> 131.7 us, M=2048 282.7 -> 245.9 us against the 4-wave kernel). The older 256 x 128
// LDS-staged kernel remains for shapes the wide kernel does not cover.
constexpr int kTiledMinM = 128;

struct W4Wide {
  WidePlan plan;
  int tn;
  int spg;  // K slabs (32 rows) per quantization group
};

// Prefetch depth of a wide W4 launch with tn-column tiles.
constexpr int w4_wide_pd(int tn) { return tn == 256 ? 4 : 2; }

// Whether the decode kernel keeps a call from 33 rows whose K ends in half an iteration of the wide tiles.
// It ran all of these up to 127 rows before the tiles took them, and above that where K is no multiple of
// the LDS-staged kernel's 128 rows. Two estimates in us, compared on 1601 calls timed on both kernels
// (M 33 to 256, K from 320 to 11136, N from 1024 to 14336; fp16 and bf16 at groups of 128, fp16 alone at 64
// and 256; decode's misses by 8% rms, the wide one's by 10%). The factor on the wide side leans to decode,
// where a miss costs more. The choice is 0.2% from the faster kernel on average and 12 calls are more
// than 4% slower than on decode (14% at most); the wide tiles alone had 489, by up to 131%
// (K=896 N=8192 M=127 bf16 8.5 -> 19.6 us).
// From 128 rows on it gives decode only short K (812 such calls of M 128 to 2048, groups of 32 and 64, both
// dtypes: 0.48 to 0.68 of the wide tiles' time on average; 16 calls 5 to 32% slower, as they were before the tiles:
// K=448 N=2048 M=768 bf16 15.3 -> 11.6 us, but K=2752 N=256 M=128 13.9 -> 18.3).
bool w4_decode_stays(int M, int N, int K, int group, bool bf16, const WidePlan& w) {
  DecodePlan d;
  if (!plan_decode(M, N, K, group / 32, &d)) return false;
  if (splitk_workspace_bytes(M, N, d.splits) > KBH_W4A16_NOALLOC_SCRATCH_BYTES) return false;  // the no-alloc entry point takes the call
  const int grid = d.ntiles * d.splits * d.mblocks;
  const float dec = (d.splits > 1 ? 5.94f : 4.1f) + 0.673f * decode_cost(M, N, d.nw, d.spw, d.waves, d.splits, grid) +
                    0.93f * (float)((grid + 255) / 256) - 0.26f * (float)d.waves;
  return dec <= 1.05f * (1.68f * w.cost + (w.tm == 64 ? -2.5f : -0.7f) + (w.splits > 1 ? 0.8f : 0.f) + (bf16 ? 0.4f : 0.f));
}

bool plan_w4_wide(int M, int N, int K, int group, bool bf16, W4Wide* w) {
  if (M < kWideMinM) return false;
  w->spg = group / 32;
  w->tn = N >= 256 ? 256 : 128;
  // 65 to 128 rows and N of 128 mod 256: 128-column tiles while their finest split (8 slabs) is at most one
  // workgroup per CU. The half column tile that the 256-column ones compute twice costs them more there
  // (bf16 M=96 2048 x 1408 13.4 against 15.2 us, 4096 x 384 13.0 / 14.7; fp16 M=96 4% and M=128 even),
  // and beyond they win at once (K x N of 8.8 M 7 to 20%, 35 M 40%).
  if (M > 64 && M <= 128 && N % 256 != 0 && K % (32 * wide_iteration(w->spg, w4_wide_pd(128))) == 0 && (long)N * K <= 256L * 128 * 256)
    w->tn = 128;
  if (M > 128 && w->tn != 256) return false;
  // Slabs per unit of K: the warp-specialised kernels (256-column tiles, x under 2 GiB) take half
  // iterations. (K = 29568 holds an odd number of 128-row groups: on the LDS-staged and decode
  // kernels, which took it before, N=8192 M=64 / 256 / 1024 ran 164 / 784 / 771 us; now 62 / 161 /
  // 518.)
  const bool ws = w->tn == 256 && (size_t)(M + 256) * K * 2 < ((size_t)1 << 31);
  const int unit = wide_iteration(w->spg, w4_wide_pd(w->tn)) / (ws ? 2 : 1);
  // Up to 64 rows with 256-column tiles: 64 x 256 tiles (2 x 2 waves of 32 x 128); a 128-row
  // tile would spend half its MFMAs and A loads on padding there. Above 128 rows the estimate
  // chooses between 128-row and 256-row tiles.
  const bool rows64 = M <= 64 && w->tn == 256;
  if (!plan_wide(M, N, K, w->tn, 32, unit, unit, w->tn == 128 ? 512 : 256, bf16 ? kBf16Costs : kHalfCosts,
                 &w->plan, rows64 ? 64 : 128))
    return false;
  return !(ws && (M < kTiledMinM || K % (TBK * TDEPTH) != 0) && K % (64 * unit) != 0 &&
           w4_decode_stays(M, N, K, group, bf16, w->plan));
}

// Calls of the wide tiles that needed no scratch before those took them (K that ends in half an
// iteration, more than 128 rows of N of 128 mod 256): without scratch they keep the LDS-staged or, on the
// workspace, the decode kernel.
bool w4_scratch_free(int M, int N, int K, int spg) {
  return (M > 128 && N % 256 != 0) || K % (32 * wide_iteration(spg, w4_wide_pd(N % 256 == 0 ? 256 : 128))) != 0;
}

// Scratch of the wide kernels, for either dtype (the query does not name it): the larger plan's.
size_t w4_wide_scratch_bytes(int M, int N, int K, int group) {
  size_t best = 0;
  for (bool bf16 : {false, true}) {
    W4Wide w;
    if (!plan_w4_wide(M, N, K, group, bf16, &w)) continue;
    const size_t b = wide_workspace_bytes(M, N, w.plan.splits);
    best = b > best ? b : best;
  }
  return best;
}

template <bool BF16, int TM, int TN, int SPG>
void launch_w4_wide(const W4Wide& w, const void* x, const int32_t* qw, const void* s, const void* z,
                    void* y, float* scratch, int M, int N, int K, int group, hipStream_t st) {
  using E = WideHalf<BF16>;
  using BP = W4WidePolicy<BF16, TN>;
  using EP = HalfOut<BF16>;
  // MFMA waves along M: 2 x 2 waves for 64- and 128-row tiles (128-row tiles: 64 x 128 per wave,
  // each B fragment read by 2 waves instead of 4; K=14336 N=4096 M=128 35.6 -> 34.9 us, M=256
  // 50.9 -> 49.8 against 4 x 1 waves of 32 x 256), 4 x 1 for the 4-wave kernel's 256-row tiles.
  constexpr int WM = TM == 256 ? 4 : 2;
  const BP bp{(const uint32_t*)qw, (const uint16_t*)s, (const uint16_t*)z, N, group, 0, 0,
              0x000F000Fu};
  const EP ep{(uint16_t*)y, N};
  // Producer sets of the warp-specialised kernel: two for 64-row tiles, whose MFMA waves need
  // only 64 accumulator registers, so that 12 waves fit (K=14336 N=4096: M=33 24.2 -> 23.5 us,
  // M=48 25.4 -> 24.7, M=64 26.7 -> 26.4; an 8-slab raw ring on top measured no faster).
  // bf16 takes two sets for 128-row tiles as well: its fp32 dequantization is about twice fp16's
  // instructions (group 128, 4096 x 4096 M=128 27.6 -> 26.6 us; the Mixtral FFN T=512 1013 -> 954);
  // fp16 is 1-3% faster with one (M=256 45.2 against 46.0).
  constexpr int PS = TM == 64 || BF16 ? 2 : 1;
  if constexpr (TM <= 128 && TN == 256) {
    // 128-row tiles stage x through LDS too (XD) while x is under 2 GiB.
    if (TM == 128 && (size_t)M * K * 2 < ((size_t)1 << 31))
      hipLaunchKernelGGL((tiled_ws_gemm<E, TM, WM, SPG, BP, EP, DenseRows, w4_wide_pd(TN), PS,
                                        TM == 128>),
                         dim3(w.plan.grid), dim3(256 * (1 + PS)), 0, st,
                         x, bp, ep, scratch, M, N, K, w.plan.sp,
                         DenseRows{M});
    else
      hipLaunchKernelGGL((tiled_ws_gemm<E, TM, WM, SPG, BP, EP, DenseRows, w4_wide_pd(TN), TM == 64 ? 2 : 1>),
                         dim3(w.plan.grid), dim3(TM == 64 ? 768 : 512), 0, st,
                         x, bp, ep, scratch, M, N, K, w.plan.sp,
                         DenseRows{M});
  } else {
    // 256 x 256 tiles: the 12-wave kernel while x is under 2 GiB (its buffer offsets are
    // 32-bit), else the 4-wave one.
    bool done = false;
    if constexpr (TM == 256 && TN == 256) {
      if ((size_t)(M + TM) * K * 2 < ((size_t)1 << 31)) {
        hipLaunchKernelGGL((tiled_ws256_gemm<E, SPG, BP, EP, w4_wide_pd(TN)>), dim3(w.plan.grid),
                           dim3(768), 0, st, x, bp, ep, scratch, M, N, K, w.plan.sp);
        done = true;
      }
    }
    if (!done)
      hipLaunchKernelGGL((tiled_wide_gemm<E, TM, WM, SPG, BP, EP, DenseRows, 0, w4_wide_pd(TN)>),
                         dim3(w.plan.grid), dim3(256), 0, st,
                         x, bp, ep, scratch, M, N, K, w.plan.sp,
                         DenseRows{M});
  }
  if (w.plan.splits > 1) {
    const size_t n4 = (size_t)M * N / 4;
    hipLaunchKernelGGL((wide_reduce_kernel<E, EP>), dim3((unsigned)((n4 + 255) / 256)), dim3(256),
                       0, st, scratch, ep, N, n4, w.plan.splits);
  }
}

template <bool BF16, int TM, int TN>
void dispatch_w4_wide_spg(const W4Wide& w, const void* x, const int32_t* qw, const void* s,
                          const void* z, void* y, float* scratch, int M, int N, int K, int group,
                          hipStream_t st) {
  switch (w.spg) {
    case 1: return launch_w4_wide<BF16, TM, TN, 1>(w, x, qw, s, z, y, scratch, M, N, K, group, st);
    case 2: return launch_w4_wide<BF16, TM, TN, 2>(w, x, qw, s, z, y, scratch, M, N, K, group, st);
    case 4: return launch_w4_wide<BF16, TM, TN, 4>(w, x, qw, s, z, y, scratch, M, N, K, group, st);
    default: return launch_w4_wide<BF16, TM, TN, 8>(w, x, qw, s, z, y, scratch, M, N, K, group, st);
  }
}

template <bool BF16>
void dispatch_w4_wide(const W4Wide& w, const void* x, const int32_t* qw, const void* s,
                      const void* z, void* y, float* scratch, int M, int N, int K, int group,
                      hipStream_t st) {
  if (w.plan.tm == 256)
    dispatch_w4_wide_spg<BF16, 256, 256>(w, x, qw, s, z, y, scratch, M, N, K, group, st);
  else if (w.plan.tm == 64)
    dispatch_w4_wide_spg<BF16, 64, 256>(w, x, qw, s, z, y, scratch, M, N, K, group, st);
  else if (w.tn == 256)
    dispatch_w4_wide_spg<BF16, 128, 256>(w, x, qw, s, z, y, scratch, M, N, K, group, st);
  else
    dispatch_w4_wide_spg<BF16, 128, 128>(w, x, qw, s, z, y, scratch, M, N, K, group, st);
}

}  // namespace

// Bytes of device memory the path a call takes needs beyond its inputs and outputs: the wide
// kernel's split-K scratch, nothing for the LDS-staged kernel, or the decode kernel's split-K
// workspace (the dispatch order of kbh_w4a16_gemm).
size_t w4a16_path_bytes(int M, int N, int K, int group, int dtype) {
  W4Wide w;
  if (plan_w4_wide(M, N, K, group, dtype == KBH_BF16, &w)) return wide_workspace_bytes(M, N, w.plan.splits);
  if (M >= kTiledMinM && K % (TBK * TDEPTH) == 0) return 0;
  DecodePlan p;
  if (!plan_decode(M, N, K, group / 32, &p)) return 0;
  return decode_workspace_bytes(p, M, N, K, group);
}

}  // namespace kbh

extern "C" size_t kbh_w4a16_workspace_bytes(int M, int N, int K, int group) {
  kbh::DecodePlan p;
  if (M < 1 || N < 128 || K < 32 || group < 32 || !kbh::plan_decode(M, N, K, group / 32, &p))
    return 0;
  return kbh::decode_workspace_bytes(p, M, N, K, group);
}

extern "C" size_t kbh_w4a16_scratch_bytes(int M, int N, int K, int group) {
  if (M < 1 || N < 128 || K < 32 || group < 32) return 0;
  return kbh::w4_wide_scratch_bytes(M, N, K, group);
}

extern "C" int kbh_w4a16_kernel(int M, int N, int K, int group, int dtype, int* splits) {
  using namespace kbh;
  if (splits) *splits = 1;
  if (M < 1 || N < 128 || K < 32 || N % 128 != 0 || !quant_group_ok(K, group)) return KBH_KERNEL_NONE;
  W4Wide w;
  if (plan_w4_wide(M, N, K, group, dtype == KBH_BF16, &w)) {
    if (splits) *splits = w.plan.splits;
    return w.tn == 128 ? KBH_KERNEL_NARROW128 : w.plan.tm;
  }
  if (M >= kTiledMinM && K % (TBK * TDEPTH) == 0) return KBH_KERNEL_STAGED;
  DecodePlan p;
  if (!plan_decode(M, N, K, group / 32, &p)) return KBH_KERNEL_NONE;
  const int s = plan_stream(p, M, N, K, group);
  if (splits) *splits = s > 0 ? s : p.splits;
  return s > 0 ? KBH_KERNEL_STREAM : KBH_KERNEL_DECODE;
}

extern "C" int kbh_w4a16_gemm(const void* x, const int32_t* qweight, const void* scales,
                              const void* zeros, void* y, void* workspace, size_t workspace_bytes,
                              void* scratch, size_t scratch_bytes, int M, int N, int K, int group,
                              int dtype, void* stream) {
  using namespace kbh;
  if (!x || !qweight || !scales || !zeros || !y) return KBH_ERR_NULL;
  if (dtype != KBH_F16 && dtype != KBH_BF16) return KBH_ERR_DTYPE;
  if (M < 1 || N < 128 || K < 32 || (N % 128) != 0 || (K % 32) != 0) return KBH_ERR_SHAPE;
  if (group != 32 && group != 64 && group != 128 && group != 256) return KBH_ERR_SHAPE;
  if (K % group != 0) return KBH_ERR_SHAPE;
  if (!aligned16(x) || !aligned16(qweight) || !aligned16(scales) || !aligned16(zeros) ||
      !aligned16(y))
    return KBH_ERR_ALIGN;
  const bool bf = dtype == KBH_BF16;
  hipStream_t st = (hipStream_t)stream;

  W4Wide wide;
  bool is_wide = plan_w4_wide(M, N, K, group, bf, &wide);
  if (is_wide) {
    const size_t need = wide_workspace_bytes(M, N, wide.plan.splits);
    if (need > 0 && (!scratch || scratch_bytes < need)) {
      if (!w4_scratch_free(M, N, K, wide.spg)) return KBH_ERR_WORKSPACE;
      is_wide = false;
    } else if (need > 0 && !aligned16(scratch)) {
      return KBH_ERR_ALIGN;
    }
  }
  if (is_wide) {
    if (bf) dispatch_w4_wide<true>(wide, x, qweight, scales, zeros, y, (float*)scratch, M, N, K, group, st);
    else dispatch_w4_wide<false>(wide, x, qweight, scales, zeros, y, (float*)scratch, M, N, K, group, st);
    return launch_status();
  }

  if (M >= kTiledMinM && K % (TBK * TDEPTH) == 0) {
    if (bf) {
      const W4SlabPolicy<true> bp{(const uint32_t*)qweight, (const uint16_t*)scales,
                                  (const uint16_t*)zeros, N, group, 0, 0};
      hipLaunchKernelGGL((tiled_f16_gemm<true, W4SlabPolicy<true>>), tiled_f16_grid(M, N),
                         dim3(256), 0, st, (const uint16_t*)x, bp, (uint16_t*)y, M, N, K);
    } else {
      const W4SlabPolicy<false> bp{(const uint32_t*)qweight, (const uint16_t*)scales,
                                   (const uint16_t*)zeros, N, group, 0, 0};
      hipLaunchKernelGGL((tiled_f16_gemm<false, W4SlabPolicy<false>>), tiled_f16_grid(M, N),
                         dim3(256), 0, st, (const uint16_t*)x, bp, (uint16_t*)y, M, N, K);
    }
    return launch_status();
  }

  DecodePlan p;
  if (!plan_decode(M, N, K, group / 32, &p)) return KBH_ERR_SHAPE;
  const int ss = plan_stream(p, M, N, K, group);  // its slices are written also when K is unsplit
  const size_t need = decode_workspace_bytes(p, M, N, K, group);
  if (need > 0 && (!workspace || workspace_bytes < need)) return KBH_ERR_WORKSPACE;
  if (need > 0 && !aligned16(workspace)) return KBH_ERR_ALIGN;
  float* acc = (float*)workspace;
  if (ss > 0) {
    if (bf) launch_dense_stream<true>(ss, x, qweight, scales, zeros, y, acc, M, N, K, group, st);
    else launch_dense_stream<false>(ss, x, qweight, scales, zeros, y, acc, M, N, K, group, st);
    return launch_status();
  }
  if (bf) dispatch_decode<true>(p, x, qweight, scales, zeros, y, acc, M, N, K, group, st);
  else dispatch_decode<false>(p, x, qweight, scales, zeros, y, acc, M, N, K, group, st);
  return launch_status();
}
