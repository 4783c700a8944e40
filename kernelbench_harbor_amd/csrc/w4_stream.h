// Streaming W4A16 kernel for up to 16 rows per tile (w4_stream_kernel): the weights of many
// workgroups' worth of K x N pass through each CU in one continuous stream.
//
// w4a16_decode_kernel (w4a16.hip) issues every load of a wave before any arithmetic and ends: where
// its grid is several workgroups per CU (large layers, the experts of a mixture), each of them
// fills the memory pipeline and drains it again. Here a wave walks its K range in 64-row chunks with
// two chunk buffers in registers: chunk i + 1's loads are issued before chunk i's MFMAs, so 8 to
// 16 KB per wave stay in flight; 4 waves and 66 KB of LDS per workgroup let two workgroups share
// a CU, one streaming while the other reduces.
//
// The arithmetic is the decode kernel's: nibbles become fp16/bf16 B operands by one v_perm_b32 and
// one v_and_or_b32 per pair (the codes on a magic exponent), one 16x16x32 MFMA per (word, nibble),
// and scale and zero point are folded into fp32 totals once per quantization group, with
// sum_k x_k from one MFMA against a ones fragment. The 4 waves of a workgroup take consecutive
// parts of its K range and meet in LDS; the workgroup stores its fp32 tile into slice `split` of the
// workspace.
//
// An infinity in x, or sums past fp32's range, leave NaN in all columns of that arithmetic (infinity
// minus infinity). On expert tiles, whose batches of 32 rows and more per expert multiply dequantized
// weights, w4_redo computes the sums of such rows once more as those kernels do.
//
// Rows: dense (tile y is rows 16 y ..) or an expert tile table of 16-row entries with x rows
// gathered through the slot permutation. Two weight matrices of one shape (gate and up) may be
// walked as one: column tiles past the first matrix's go to the second.
#pragma once

#include "kbh_common.h"
#include "splitk.h"
#include "w4_dequant.h"

namespace kbh {

constexpr int kStreamWaves = 4;
constexpr int kStreamCols = 256;       // output columns of one workgroup
constexpr int kStreamChunk = 64;       // K rows per chunk (two MFMA steps)

struct W4Mat {
  const uint32_t* qw;
  const uint16_t* scales;
  const uint16_t* zeros;
};

struct W4StreamArgs {
  const uint16_t* x;
  W4Mat mat[2];
  float* slices;       // [splits][M][ld]
  const int* tiles;    // grouped: {expert, first slot, rows} per 16-row entry
  const int* perm;     // grouped: slot -> 2 * token + k
  size_t q_stride, s_stride;  // elements between experts
  int M, ld;           // rows and columns of one slice
  int N, K, group;     // of one matrix
  int splits;
  int tiles0;          // column tiles of one matrix
  int gather;          // grouped: x row perm[slot] / 2 (else the slot), output row the slot
                       // (else perm[slot])
};

// A wave's sums in LDS (column set 8 w + nib, rows 4 g + i of lane 16 g + c) again where they are not
// finite, over K rows [k0, k1): the x row of slot s0 + that row (by way of perm, unless null) times the
// weights dequantized as the reference and the wide tiles do it (q - z and the product with s each rounded once), so that an infinity meets each
// weight's sign (and a zero weight gives NaN). One K row at a time and nothing unrolled: it is rare, and
// costs the kernel no registers.
template <bool BF16, int NCS>
__device__ inline void w4_redo(float* slice, int rows, const uint16_t* x, int s0, const int* perm, const uint32_t* qw,
                               const uint16_t* sp, const uint16_t* zp, int N, int K, int group, int k0, int k1) {
  const int lane = threadIdx.x & 63, g4 = 4 * (lane >> 4);
  const auto round = [](float v) { return half_bits_to_f32<BF16>(f32_to_half_bits<BF16>(keep_f32(v))); };
#pragma unroll 1
  for (int i = 0; i < 4; ++i) {
    if (g4 + i >= rows) break;
    const uint16_t* xr = x + (size_t)(perm ? perm[s0 + g4 + i] >> 1 : s0 + g4 + i) * K;
#pragma unroll 1
    for (int cs = 0; cs < NCS; ++cs) {
      float& t = slice[cs * kSplitKCsStride + lane * 4 + i];
      if (__builtin_isfinite(t)) continue;
      float v = 0.f;
#pragma unroll 1
      for (int k = k0; k < k1; ++k) {
        const size_t o = (size_t)(k / group) * N + cs;
        const float q = (float)((qw[(size_t)k * (N >> 3) + (cs >> 3)] >> (4 * (cs & 7))) & 15u);
        v = fmaf(half_bits_to_f32<BF16>(xr[k]), round(round(q - half_bits_to_f32<BF16>(zp[o])) * half_bits_to_f32<BF16>(sp[o])), v);
      }
      t = v;
    }
  }
}

// SPG: K steps (32 rows) per quantization group: 1, 2, 4 or 8.
template <int SPG, bool BF16, bool GROUPED>
__global__ __launch_bounds__(64 * kStreamWaves, 2) void w4_stream_kernel(W4StreamArgs a) {
  constexpr int NW = 2, NCS = 8 * NW;
  constexpr uint32_t MAGIC = BF16 ? kMagicBF16 : kMagicF16;
  constexpr int CPG = SPG > 2 ? SPG / 2 : 1;  // chunks per unit (a group, at least one chunk)
  constexpr int GPC = SPG == 1 ? 2 : 1;       // groups per chunk
  __shared__ SplitKSmem<NCS, float, kStreamWaves> sm;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int id = xcd_remap(blockIdx.x, gridDim.x);
  const int tile = id / a.splits, split = id - tile * a.splits;
  int expert = 0, s0 = 16 * (int)blockIdx.y, rows = a.M - s0;
  if constexpr (GROUPED) {
    const int* tl = a.tiles + 3 * blockIdx.y;
    expert = tl[0];
    s0 = tl[1];
    rows = tl[2];
    if (rows <= 0) return;  // unused table entry (uniform across the workgroup)
  }
  rows = min(rows, 16);
  const bool second = tile >= a.tiles0;
  const W4Mat& mt = a.mat[second ? 1 : 0];
  const int n0 = (tile - (second ? a.tiles0 : 0)) * kStreamCols;
  const int N = a.N, K = a.K, NP = N >> 3;
  // This wave's units of K (consecutive parts of the split's range, uneven where they must be).
  const int units = K / (CPG * kStreamChunk);
  const int ub = (int)((long)units * split / a.splits), ue = (int)((long)units * (split + 1) / a.splits);
  const int wb = ub + (ue - ub) * wave / kStreamWaves, we = ub + (ue - ub) * (wave + 1) / kStreamWaves;

  // Rows past the tile re-read its first row: an output row depends on its own x row alone, and
  // theirs are never stored.
  int src = s0 + (c < rows ? c : 0);
  if constexpr (GROUPED)
    if (a.gather) src = a.perm[src] >> 1;

  const uint32_t* qw = mt.qw + (size_t)expert * a.q_stride;
  const __amdgpu_buffer_rsrc_t qres = make_rsrc(qw, (size_t)K * NP * 4);
  const uint32_t qlane = (uint32_t)(8 * g * NP + (n0 >> 3) + c * NW) * 4u;
  const uint16_t* sp = mt.scales + (size_t)expert * a.s_stride + n0 + 8 * c * NW;
  const uint16_t* zp = mt.zeros + (size_t)expert * a.s_stride + n0 + 8 * c * NW;
  const uint16_t* xp = a.x + (size_t)src * K + 8 * g;

  struct Chunk {
    kbh_u32x2 w[2][8];
    kbh_u32x4 x[2];
  };
  struct Consts {
    kbh_u32x4 s[GPC][NW], z[GPC][NW];
  };
  const int cb = wb * CPG, ce = we * CPG;  // this wave's chunks
  auto load = [&](Chunk& ch, int i) {
    const int k0 = min(i, ce - 1) * kStreamChunk;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 8; ++r)
        ch.w[u][r] = __builtin_bit_cast(
            kbh_u32x2, __builtin_amdgcn_raw_buffer_load_b64(qres, qlane, (k0 + 32 * u + r) * NP * 4, kBufNT));
#pragma unroll
    for (int u = 0; u < 2; ++u) ch.x[u] = *reinterpret_cast<const kbh_u32x4*>(xp + k0 + 32 * u);
  };
  // Constants of the group(s) that end in chunk i.
  auto load_consts = [&](Consts& cs, int i) {
    const int gi = min(i, ce - 1) * kStreamChunk / a.group;
#pragma unroll
    for (int q = 0; q < GPC; ++q)
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        cs.s[q][w] = *reinterpret_cast<const kbh_u32x4*>(sp + (size_t)(gi + q) * N + 8 * w);
        cs.z[q][w] = *reinterpret_cast<const kbh_u32x4*>(zp + (size_t)(gi + q) * N + 8 * w);
      }
  };

  const uint32_t one = BF16 ? kOneBF16 : kOneF16;
  const kbh_u32x4 ones = {one, one, one, one};
  uint32_t mlo = 0x000F000Fu, mhi = 0x00F000F0u, magic = MAGIC;
  asm volatile("" : "+s"(mlo), "+s"(mhi));
  asm volatile("" : "+v"(magic));
  kbh_f32x4 tot[NCS], part[NCS], xs = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int cs = 0; cs < NCS; ++cs) {
    tot[cs] = kbh_f32x4{0.f, 0.f, 0.f, 0.f};
    part[cs] = tot[cs];
  }
  auto step = [&](const Chunk& ch, int u) {
    xs = mfma16x16x32<BF16>(ch.x[u], ones, xs);
#pragma unroll
    for (int w = 0; w < NW; ++w)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        kbh_u32x4 blo, bhi;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          const uint32_t P = pair_bytes_rt(ch.w[u][2 * p][w], ch.w[u][2 * p + 1][w], j);
          blo[p] = (P & mlo) | magic;
          bhi[p] = BF16 ? (((P >> 4) & mlo) | magic) : ((P & mhi) | magic);
        }
        part[w * 8 + 2 * j] = mfma16x16x32<BF16>(ch.x[u], blo, part[w * 8 + 2 * j]);
        part[w * 8 + 2 * j + 1] = mfma16x16x32<BF16>(ch.x[u], bhi, part[w * 8 + 2 * j + 1]);
      }
  };
  auto fold = [&](const Consts& cs, int q) {
#pragma unroll
    for (int w = 0; w < NW; ++w)
#pragma unroll
      for (int nib = 0; nib < 8; ++nib) {
        const float s = half_bits_to_f32<BF16>(half_of(cs.s[q][w], nib));
        const float z = half_bits_to_f32<BF16>(half_of(cs.z[q][w], nib));
        const float f = (!BF16 && (nib & 1)) ? 0.0625f : 1.0f;
        const float bz = (BF16 ? 128.0f : ((nib & 1) ? 64.0f : 1024.0f)) + z;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float t = fmaf(-bz, xs[i], part[w * 8 + nib][i] * f);
          tot[w * 8 + nib][i] = fmaf(s, t, tot[w * 8 + nib][i]);
        }
        part[w * 8 + nib] = kbh_f32x4{0.f, 0.f, 0.f, 0.f};
      }
    xs = kbh_f32x4{0.f, 0.f, 0.f, 0.f};
  };

  // Two chunk buffers; the loop body covers two chunks, or a whole unit when that is more, so
  // that buffers and fold points are static. A unit of one chunk (groups of 32 or 64 rows) may
  // leave a single chunk over. Loads past the range re-read its last chunk (never used).
  constexpr int BODY = CPG > 2 ? CPG : 2;
  if (cb < ce) {
    Chunk buf[2];
    Consts cs;
    load(buf[0], cb);
    auto one_chunk = [&](auto idx, int i) {
      constexpr int u = decltype(idx)::value;
      constexpr bool ends = (u + 1) % CPG == 0;  // a group ends in this chunk
      if constexpr (ends) load_consts(cs, i);
      load(buf[(u + 1) & 1], i + 1);
      __builtin_amdgcn_sched_barrier(0);  // the next chunk's loads go out before this one's math
      step(buf[u & 1], 0);
      if constexpr (SPG == 1) fold(cs, 0);
      step(buf[u & 1], 1);
      if constexpr (ends) fold(cs, GPC - 1);
      __builtin_amdgcn_sched_barrier(0);
    };
    int i = cb;
    for (; i + BODY <= ce; i += BODY) {
      one_chunk(WideIdx<0>{}, i);
      one_chunk(WideIdx<1>{}, i + 1);
      if constexpr (BODY == 4) {
        one_chunk(WideIdx<2>{}, i + 2);
        one_chunk(WideIdx<3>{}, i + 3);
      }
    }
    if constexpr (CPG == 1)
      if (i < ce) one_chunk(WideIdx<0>{}, i);
  }
#pragma unroll
  for (int cs = 0; cs < NCS; ++cs) asm volatile("" : "+v"(tot[cs]));
  float* slice = a.slices + (size_t)split * a.M * a.ld + (size_t)tile * kStreamCols;
  const auto store = [&](int r, int n, float v) {
    int row = s0 + r;
    if constexpr (GROUPED)
      if (!a.gather) row = a.perm[row];
    slice[(size_t)row * a.ld + n] = v;
  };
  if constexpr (GROUPED) {
    bool redo = false;
#pragma unroll
    for (int cs = 0; cs < NCS; ++cs)
#pragma unroll
      for (int i = 0; i < 4; ++i) redo |= !__builtin_isfinite(tot[cs][i]);
    const bool any = __any(redo);
    splitk_wave_sum<NCS, float, kbh_f32x4>(tot, sm, rows, store, [&](float* mine) {
      if (any)
        w4_redo<BF16, NCS>(mine, rows, a.x, s0, a.gather ? a.perm : nullptr, qw + (n0 >> 3) + c * NW, sp, zp, N, K, a.group,
                           cb * kStreamChunk, ce * kStreamChunk);
    });
  } else {
    splitk_wave_sum<NCS, float, kbh_f32x4>(tot, sm, rows, store);
  }
}

// Whether the kernel takes K x N matrices of this group size (32-bit buffer offsets, whole units).
inline bool w4_stream_ok(int N, int K, int group) {
  const int unit = group > kStreamChunk ? group : kStreamChunk;
  return N % kStreamCols == 0 && K % unit == 0 && (size_t)K * N / 2 < ((size_t)1 << 31);
}

// Estimated cost (decode_cost's units in w4a16.hip) of `row_tiles` row tiles of M rows in all on
// `mats` K x N matrices split s ways: the weight KB a CU streams, one workgroup after another at
// 22.5 KB per unit (a second round beside the first gains nothing: dense K=29568 N=8192 M=16 128 /
// 256 / 448 workgroups 50.1 / 34.2 / 37.2 us; eight waves per workgroup measured the same) with a
// fixed cost of its own, and the fp32 slices written and read.
inline float w4_stream_cost(int M, int N, int K, int row_tiles, int mats, int s) {
  const long wgs = (long)(N / kStreamCols) * row_tiles * mats * s;
  const float kb = (float)K / s * (kStreamCols / 2048.0f);  // of one workgroup
  return 3.7f + (float)((wgs + 255) / 256) * (1.0f + kb / 22.5f) + (float)s * M * N * mats * 8.0f / 1024.0f / 2540.0f;
}

// The K split of least estimated cost with at least one unit of K per wave.
inline int w4_stream_splits(int M, int N, int K, int group, int row_tiles, int mats) {
  const int unit = group > kStreamChunk ? group : kStreamChunk;
  const int most = K / unit / kStreamWaves;
  int best = 1;
  float c = w4_stream_cost(M, N, K, row_tiles, mats, 1);
  for (int s = 2; s <= most && s <= 64; ++s) {
    const float cs = w4_stream_cost(M, N, K, row_tiles, mats, s);
    if (cs < c) {
      c = cs;
      best = s;
    }
  }
  return best;
}

template <bool BF16, bool GROUPED>
void launch_w4_stream(const W4StreamArgs& a, int col_tiles, int row_tiles, hipStream_t st) {
  const dim3 grid((unsigned)(col_tiles * a.splits), (unsigned)row_tiles), block(64 * kStreamWaves);
  switch (a.group / 32) {
    case 1: hipLaunchKernelGGL((w4_stream_kernel<1, BF16, GROUPED>), grid, block, 0, st, a); return;
    case 2: hipLaunchKernelGGL((w4_stream_kernel<2, BF16, GROUPED>), grid, block, 0, st, a); return;
    case 4: hipLaunchKernelGGL((w4_stream_kernel<4, BF16, GROUPED>), grid, block, 0, st, a); return;
    default: hipLaunchKernelGGL((w4_stream_kernel<8, BF16, GROUPED>), grid, block, 0, st, a); return;
  }
}

}  // namespace kbh
