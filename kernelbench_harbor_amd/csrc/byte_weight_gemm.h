// Byte-weight GEMM for gfx950: y = x @ W with W[k, n] = dtype(decode(w[k, n]) * scales[k/B, n]),
// w one byte per element, [K, N] with N contiguous, one scale per B consecutive k of a column.
// Decoders (DEC): kDecE4M3 — OCP e4m3fn codes with fp16 scales (tasks/fp8_microscale/
// fp8_microscale__llama3_8b_down__b128__fp16/environment/reference.py:9-12); kDecInt8 — int8
// values (int4 stored one per byte) with scales in the activation dtype (tasks/multi_lora_qgemm/
// multi_lora_qgemm__llama3_8b_r16__fp16/environment/reference.py:12). Either way every weight
// is rounded once, as in the references: the decoded value is exact in fp16/bf16 and fp32, and
// the product with the scale is rounded once (v_pk_mul_f16, or an exact fp32 product rounded to
// bf16).
//
// The decode and LDS-staged kernels transpose 4x4 byte blocks in registers so that each lane holds
// consecutive k of one column, as the MFMA B operand needs; the others pair rows by v_perm_b32.
//  * byte_decode_kernel (small M): a wave owns 128 columns (8 per lane, dwordx2 loads) and SPW
//    steps of 32 k for MB blocks of 16 rows (each dequantised weight fragment feeds MB MFMAs, so
//    the weights are streamed once per 16 MB rows); all loads up front; 16x16x32 fp16/bf16
//    MFMAs; split-K epilogue of splitk.h, once per row block.
//  * byte_stream_kernel (e4m3, up to 16 rows, layers whose decode grid is over two workgroups per CU):
//    the same tile, K walked in a continuous stream.
//  * larger M: the warp-specialised wide tiles (tiled_ws.h, tiled_ws256.h) with ByteWidePolicy, or
//    tiled_f16_gemm (tiled_f16.h) with ByteSlabPolicy for shapes they do not cover.
#pragma once

#include "kbh_common.h"
#include "splitk.h"
#include "tiled_f16.h"
#include "tiled_ws.h"
#include "tiled_ws256.h"
#include "w4_dequant.h"

namespace kbh {
namespace {

constexpr int kDecE4M3 = 0;
constexpr int kDecInt8 = 1;

typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef float f2_t __attribute__((ext_vector_type(2)));

// 4x4 byte transpose: r[i] holds bytes (row i, columns 0..3); c[j] receives (rows 0..3, column j).
__device__ inline void transpose4x4_b(const uint32_t r[4], uint32_t c[4]) {
  const uint32_t t0 = __builtin_amdgcn_perm(r[1], r[0], 0x05010400u);
  const uint32_t t1 = __builtin_amdgcn_perm(r[1], r[0], 0x07030602u);
  const uint32_t t2 = __builtin_amdgcn_perm(r[3], r[2], 0x05010400u);
  const uint32_t t3 = __builtin_amdgcn_perm(r[3], r[2], 0x07030602u);
  c[0] = __builtin_amdgcn_perm(t2, t0, 0x05040100u);
  c[1] = __builtin_amdgcn_perm(t2, t0, 0x07060302u);
  c[2] = __builtin_amdgcn_perm(t3, t1, 0x05040100u);
  c[3] = __builtin_amdgcn_perm(t3, t1, 0x07060302u);
}

// Four codes (bytes of v, k order) times scale s -> four dtype values in two dwords, each
// rounded once. e4m3: s holds fp16 bits; int8: s holds bits of the activation dtype.
template <bool BF16, int DEC>
__device__ inline kbh_u32x2 byte4_dequant(uint32_t v, uint16_t s) {
  if constexpr (DEC == kDecInt8) {
    if constexpr (BF16) {
      const float sf = bf16_bits_to_f32(s);
      const float q0 = (float)(int8_t)(v & 0xffu), q1 = (float)(int8_t)((v >> 8) & 0xffu);
      const float q2 = (float)(int8_t)((v >> 16) & 0xffu), q3 = (float)(int8_t)(v >> 24);
      return kbh_u32x2{f32x2_to_bf16x2_bits(keep_f32(q0 * sf), keep_f32(q1 * sf)),
                       f32x2_to_bf16x2_bits(keep_f32(q2 * sf), keep_f32(q3 * sf))};
    } else {
      // (byte ^ 0x80) | 0x6400 is the fp16 1024 + (q + 128); minus 1152 gives q exactly
      const _Float16 sh = __builtin_bit_cast(_Float16, s);
      const _Float16 bias = (_Float16)1152.0f;
      const uint32_t p0 = (__builtin_amdgcn_perm(0u, v, 0x0c010c00u) ^ 0x00800080u) | 0x64006400u;
      const uint32_t p1 = (__builtin_amdgcn_perm(0u, v, 0x0c030c02u) ^ 0x00800080u) | 0x64006400u;
      const h2_t lo = (__builtin_bit_cast(h2_t, p0) - h2_t{bias, bias}) * h2_t{sh, sh};
      const h2_t hi = (__builtin_bit_cast(h2_t, p1) - h2_t{bias, bias}) * h2_t{sh, sh};
      return kbh_u32x2{__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi)};
    }
  } else if constexpr (BF16) {
    const float sf = f16_bits_to_f32(s);
    const f2_t lo = __builtin_amdgcn_cvt_pk_f32_fp8(v, false);
    const f2_t hi = __builtin_amdgcn_cvt_pk_f32_fp8(v, true);
    return kbh_u32x2{f32x2_to_bf16x2_bits(keep_f32(lo[0] * sf), keep_f32(lo[1] * sf)),
                     f32x2_to_bf16x2_bits(keep_f32(hi[0] * sf), keep_f32(hi[1] * sf))};
  } else {
    const _Float16 sh = __builtin_bit_cast(_Float16, s);
    const h2_t lo = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(v, 1.0f, false) * h2_t{sh, sh};
    const h2_t hi = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(v, 1.0f, true) * h2_t{sh, sh};
    return kbh_u32x2{__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi)};
  }
}

// Side work that shares a decode launch: `blocks` further workgroups along grid.x (those of
// blockIdx.y 0) call run(index). None by default.
struct NoSide {
  static constexpr bool kAny = false;
  int blocks = 0;
  __device__ void run(int) const {}
};

template <int SPW, bool BF16, int DEC, int MB, class SIDE>
__global__ __launch_bounds__(kSplitKMaxWaves * 64) void byte_decode_kernel(
    const uint16_t* __restrict__ x, const uint8_t* __restrict__ w,
    const uint16_t* __restrict__ scales, uint16_t* __restrict__ y, float* __restrict__ acc,
    int M, int N, int K, int block, int splits, SIDE side) {
  constexpr int NCS = 8;  // lane column c owns output columns n0 + 8c .. +7
  constexpr int NWG = 128;
  __shared__ SplitKSmem<NCS, float> sm;
  const int nblocks = SIDE::kAny ? gridDim.x - side.blocks : gridDim.x;  // the GEMM's
  if constexpr (SIDE::kAny) {
    if ((int)blockIdx.x >= nblocks) {  // uniform across the workgroup
      if (blockIdx.y == 0) side.run(blockIdx.x - nblocks);
      return;
    }
  }
  const int waves = blockDim.x >> 6;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = lane & 15, g = lane >> 4;
  const int id = xcd_remap(blockIdx.x, nblocks);
  const int tile = id / splits, split = id - tile * splits;
  const int n0 = tile * NWG;
  const int m0 = blockIdx.y * 16 * MB;
  const int st0 = (split * waves + wave) * SPW;  // first 32-deep K step of this wave

  // lane (c, g): rows k0 + 8g + i (i < 8), bytes n0 + 8c .. +7
  kbh_u32x2 wd[SPW][8];
  const uint8_t* wb = w + (size_t)(st0 * 32 + 8 * g) * N + n0 + 8 * c;
#pragma unroll
  for (int u = 0; u < SPW; ++u)
#pragma unroll
    for (int i = 0; i < 8; ++i)
      wd[u][i] = __builtin_nontemporal_load(reinterpret_cast<const kbh_u32x2*>(wb + (size_t)(u * 32 + i) * N));
  kbh_u32x4 af[SPW][MB], sv[SPW];
  bool xok[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    xok[mb] = m0 + 16 * mb + c < M;
    const uint16_t* xb = x + (size_t)(xok[mb] ? m0 + 16 * mb + c : 0) * K + st0 * 32 + 8 * g;
#pragma unroll
    for (int u = 0; u < SPW; ++u) af[u][mb] = *reinterpret_cast<const kbh_u32x4*>(xb + u * 32);
  }
#pragma unroll
  for (int u = 0; u < SPW; ++u)
    sv[u] = *reinterpret_cast<const kbh_u32x4*>(scales + (size_t)(((st0 + u) * 32) / block) * N + n0 + 8 * c);
  // All loads are issued before any use (a consumer between them stalls the stream).
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < SPW; ++u)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
      if (!xok[mb]) af[u][mb] = kbh_u32x4{0u, 0u, 0u, 0u};  // rows past M contribute zero

  kbh_f32x4 part[MB][NCS];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int cs = 0; cs < NCS; ++cs) part[mb][cs] = kbh_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < SPW; ++u) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {  // dword h: columns 4h .. 4h+3
      uint32_t col[4][2];          // col[j][b]: column 4h+j, rows 4b .. 4b+3
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const uint32_t r[4] = {wd[u][4 * b][h], wd[u][4 * b + 1][h], wd[u][4 * b + 2][h],
                               wd[u][4 * b + 3][h]};
        uint32_t t4[4];
        transpose4x4_b(r, t4);
#pragma unroll
        for (int j = 0; j < 4; ++j) col[j][b] = t4[j];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int cs = 4 * h + j;
        const uint16_t s = half_of(sv[u], cs);
        const kbh_u32x2 lo = byte4_dequant<BF16, DEC>(col[j][0], s);
        const kbh_u32x2 hi = byte4_dequant<BF16, DEC>(col[j][1], s);
        const kbh_u32x4 bf = {lo[0], lo[1], hi[0], hi[1]};
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) part[mb][cs] = mfma16x16x32<BF16>(af[u][mb], bf, part[mb][cs]);
      }
    }
  }
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int mr = m0 + 16 * mb;
    const int rows = min(16, M - mr);
    if (rows <= 0) break;      // uniform across the workgroup
    if (mb) __syncthreads();   // the previous block's LDS reads are done
    splitk_reduce<NCS, float>(part[mb], sm, acc, split, splits, rows, M, N, mr, n0, [&](int r, int n, float v) {
      y[(size_t)(mr + r) * N + n0 + n] = f32_to_half_bits<BF16>(v);
    });
  }
}

// Weight-slab producer for tiled_f16_gemm: thread t loads rows 4*(t/32) .. +3 of the slab for
// columns 4*(t%32) .. +3, transposes, dequantizes and stores them k-major per column.
template <bool BF16, int DEC>
struct ByteSlabPolicy {
  const uint8_t* w;
  const uint16_t* scales;
  int N, block;
  struct Regs {
    uint32_t b[4];
    kbh_u32x2 s;
  };
  __device__ void load(Regs& r, int k0, int n0, int t) const {
    const int cq = t & 31, rq = t >> 5;
    const uint8_t* p = w + (size_t)(k0 + 4 * rq) * N + n0 + 4 * cq;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      r.b[i] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(p + (size_t)i * N));
    r.s = *reinterpret_cast<const kbh_u32x2*>(scales + (size_t)(k0 / block) * N + n0 + 4 * cq);
  }
  __device__ void store(const Regs& r, uint16_t* Bs, int t) const {
    const int cq = t & 31, rq = t >> 5;
    uint32_t cols[4];
    transpose4x4_b(r.b, cols);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint16_t s = (uint16_t)((j & 1) ? (r.s[j >> 1] >> 16) : (r.s[j >> 1] & 0xffffu));
      *reinterpret_cast<kbh_u32x2*>(&Bs[tld_row(4 * cq + j) * TLD + 4 * rq]) = byte4_dequant<BF16, DEC>(cols[j], s);
    }
  }
};

// Rows (k, k+1) of column J of a 4-column dword pair (a: row k, b: row k+1), times scale bits s:
// one dword of two dtype values, each rounded once (the arithmetic of byte4_dequant).
template <bool BF16, int DEC, int J>
__device__ inline uint32_t byte_pair_dequant(uint32_t a, uint32_t b, uint16_t s) {
  if constexpr (DEC == kDecInt8) {
    if constexpr (BF16) {
      const float sf = bf16_bits_to_f32(s);
      const float qa = (float)(int8_t)((a >> (8 * J)) & 0xffu), qb = (float)(int8_t)((b >> (8 * J)) & 0xffu);
      return f32x2_to_bf16x2_bits(qa * sf, qb * sf);
    } else {
      // byte ^ 0x6480 is the fp16 1024 + (q + 128); minus 1152 gives q exactly
      const _Float16 sh = __builtin_bit_cast(_Float16, s);
      const _Float16 bias = (_Float16)1152.0f;
      const h2_t q = __builtin_bit_cast(h2_t, pair_bytes<J>(a, b) ^ 0x64806480u) - h2_t{bias, bias};
      return __builtin_bit_cast(uint32_t, q * h2_t{sh, sh});
    }
  } else {
    // columns 0, 1 (or 2, 3) of both rows as two 16-bit halves (k, k+1)
    const uint32_t P = __builtin_amdgcn_perm(b, a, J < 2 ? 0x05010400u : 0x07030602u);
    if constexpr (BF16) {
      const float sf = f16_bits_to_f32(s);
      const f2_t v = __builtin_amdgcn_cvt_pk_f32_fp8(P, (J & 1) != 0);
      return f32x2_to_bf16x2_bits(v[0] * sf, v[1] * sf);
    } else {
      const _Float16 sh = __builtin_bit_cast(_Float16, s);
      return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(P, 1.0f, (J & 1) != 0) * h2_t{sh, sh});
    }
  }
}

// Streaming form for up to 16 rows (e4m3 weights), where the decode kernel's grid does not fit the
// GPU at once: its workgroups fill the memory pipeline, drain it, and leave a last round that is
// mostly empty. Here a wave walks its K range in 64-row chunks with two chunk buffers in registers
// (chunk i + 1's loads go out before chunk i's MFMAs, 8 to 16 KB per wave in flight), 4 waves and
// 33 KB of LDS per workgroup, so that all the workgroups of the plan are resident together and
// stream until their K range ends, with fewer slices. Two-row pairs come from v_perm_b32 as in
// ByteWidePolicy. HBM bound; e4m3 x fp16, back to back on rotating weights, against the decode kernel: 3584 x
// 18944 M=1 / 16 19.4 / 22.1 -> 17.7 / 20.8 us, 18944 x 3584 20.4 / 25.3 -> 19.2 / 20.7, 28672 x 8192 M=16
// 58.0 -> 48.3 (235 MB at 4.9 TB/s), 11008 x 4096 17.9 / 24.4 -> 14.0 / 15.6.
constexpr int kByteStreamWaves = 4;
constexpr int kByteStreamChunk = 64;  // K rows (two MFMA steps)

template <bool BF16>
__global__ __launch_bounds__(64 * kByteStreamWaves, 3) void byte_stream_kernel(
    const uint16_t* __restrict__ x, const uint8_t* __restrict__ w,
    const uint16_t* __restrict__ scales, uint16_t* __restrict__ y, float* __restrict__ acc,
    int M, int N, int K, int block, int splits) {
  constexpr int NCS = 8;  // lane column c owns output columns n0 + 8c .. +7
  __shared__ SplitKSmem<NCS, float, kByteStreamWaves> sm;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int c = lane & 15, g = lane >> 4;
  const int id = xcd_remap(blockIdx.x, gridDim.x);
  const int tile = id / splits, split = id - tile * splits;
  const int n0 = tile * 128;
  // This wave's chunks: consecutive parts of the split's, uneven where they must be.
  const int chunks = K / kByteStreamChunk;
  const int sb = (int)((long)chunks * split / splits), se = (int)((long)chunks * (split + 1) / splits);
  const int cb = sb + (se - sb) * wave / kByteStreamWaves;
  const int ce = sb + (se - sb) * (wave + 1) / kByteStreamWaves;

  const __amdgpu_buffer_rsrc_t wres = make_rsrc(w, (size_t)K * N);
  const uint32_t wlane = (uint32_t)(8 * g * N + n0 + 8 * c);
  // Rows past M re-read row 0: an output row depends on its own x row alone, and theirs are
  // never stored.
  const uint16_t* xp = x + (size_t)(c < M ? c : 0) * K + 8 * g;
  const uint16_t* sp = scales + n0 + 8 * c;
  struct Chunk {
    kbh_u32x2 w[2][8];
    kbh_u32x4 x[2], s[2];
  };
  auto load = [&](Chunk& ch, int i) {  // past the range: its last chunk again (never used)
    const int k0 = min(i, ce - 1) * kByteStreamChunk;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 8; ++r)
        ch.w[u][r] = __builtin_bit_cast(
            kbh_u32x2, __builtin_amdgcn_raw_buffer_load_b64(wres, wlane, (k0 + 32 * u + r) * N, kBufNT));
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      ch.x[u] = *reinterpret_cast<const kbh_u32x4*>(xp + k0 + 32 * u);
      ch.s[u] = *reinterpret_cast<const kbh_u32x4*>(sp + (size_t)((k0 + 32 * u) / block) * N);
    }
  };
  kbh_f32x4 part[NCS];
#pragma unroll
  for (int cs = 0; cs < NCS; ++cs) part[cs] = kbh_f32x4{0.f, 0.f, 0.f, 0.f};
  auto compute = [&](const Chunk& ch) {
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h) {  // dword h: columns 4h .. 4h+3
        kbh_u32x4 b[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) {  // rows 2p, 2p + 1
          const uint32_t a0 = ch.w[u][2 * p][h], a1 = ch.w[u][2 * p + 1][h];
          b[0][p] = byte_pair_dequant<BF16, kDecE4M3, 0>(a0, a1, half_of(ch.s[u], 4 * h + 0));
          b[1][p] = byte_pair_dequant<BF16, kDecE4M3, 1>(a0, a1, half_of(ch.s[u], 4 * h + 1));
          b[2][p] = byte_pair_dequant<BF16, kDecE4M3, 2>(a0, a1, half_of(ch.s[u], 4 * h + 2));
          b[3][p] = byte_pair_dequant<BF16, kDecE4M3, 3>(a0, a1, half_of(ch.s[u], 4 * h + 3));
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) part[4 * h + j] = mfma16x16x32<BF16>(ch.x[u], b[j], part[4 * h + j]);
      }
  };
  if (cb < ce) {
    Chunk buf[2];
    load(buf[0], cb);
    int i = cb;
    for (; i + 2 <= ce; i += 2) {
      load(buf[1], i + 1);
      __builtin_amdgcn_sched_barrier(0);  // the next chunk's loads go out before this one's math
      compute(buf[0]);
      __builtin_amdgcn_sched_barrier(0);
      load(buf[0], i + 2);
      __builtin_amdgcn_sched_barrier(0);
      compute(buf[1]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (i < ce) compute(buf[0]);
  }
  splitk_wave_sum<NCS, float, kbh_f32x4>(part, sm, min(M, 16), [&](int r, int n, float v) {
    if (splits == 1)
      y[(size_t)r * N + n0 + n] = f32_to_half_bits<BF16>(v);
    else
      acc[((size_t)split * M + r) * N + n0 + n] = v;
  });
}

// Weight producer of the warp-specialised kernels (32 rows x 256 columns per slab). Thread t owns
// rows 4rb .. 4rb+3 of columns 8cb .. 8cb+7 (the F16WidePolicy / W8WidePolicy thread map, whose
// 8-byte LDS writes are bank-conflict free; the 4-byte ones of two producer sets are not, 12 k cycles per
// workgroup at bf16 M=300 K=14336 N=4096, and still gain by the second set): four 8-byte loads, and per column its 4 consecutive K values
// as one 8-byte piece of the K-contiguous operand layout (wide_b_offset). The two-row pairs come
// straight from v_perm_b32 on two rows (no 4x4 byte transpose): the e4m3 conversions take either
// 16-bit half of a dword.
template <bool BF16, int DEC>
struct ByteWidePolicy {
  static constexpr int kTN = 256;
  static constexpr bool kHasFast = false;
  const uint8_t* w;
  const uint16_t* scales;
  int N, block;
  struct Raw {
    kbh_u32x2 r[4];
  };
  struct RawHalf {
    kbh_u32x2 r[2];
  };
  struct Grp {
    kbh_u32x4 s;
  };
  struct ScanPre {};
  __device__ ByteWidePolicy at_expert(int) const { return *this; }
  __device__ static int cb_of(int t) { return (t & 7) | (((t >> 4) & 3) << 3); }
  __device__ static int rb_of(int t) { return ((t >> 3) & 1) | ((t >> 6) << 1); }
  __device__ void load(Raw& r, int k0, int n0, int t) const {
    const uint8_t* p = w + (size_t)(k0 + 4 * rb_of(t)) * N + n0 + 8 * cb_of(t);
#pragma unroll
    for (int i = 0; i < 4; ++i)  // cached: the row blocks of a K range share them in L2
      r.r[i] = *reinterpret_cast<const kbh_u32x2*>(p + (size_t)i * N);
  }
  // Two producer sets: set `half` takes rows 4rb + 2 half, +1.
  __device__ void load_half(RawHalf& r, int k0, int n0, int t, int half) const {
    const uint8_t* p = w + (size_t)(k0 + 4 * rb_of(t) + 2 * half) * N + n0 + 8 * cb_of(t);
    r.r[0] = *reinterpret_cast<const kbh_u32x2*>(p);
    r.r[1] = *reinterpret_cast<const kbh_u32x2*>(p + N);
  }
  __device__ void load_group(Grp& g, int k0, int n0, int t) const {
    g.s = *reinterpret_cast<const kbh_u32x4*>(scales + (size_t)(k0 / block) * N + n0 + 8 * cb_of(t));
  }
  template <bool FAST>
  __device__ void prepare_group(Grp&) const {}
  // Values of column c of rows (2i, 2i+1) for NI row pairs, all columns.
  template <int NI, class R>
  __device__ void dequant(const R& r, const Grp& g, uint32_t (&v)[8][NI]) const {
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const uint32_t a = r.r[2 * i][h], b = r.r[2 * i + 1][h];
        v[4 * h + 0][i] = byte_pair_dequant<BF16, DEC, 0>(a, b, half_of(g.s, 4 * h + 0));
        v[4 * h + 1][i] = byte_pair_dequant<BF16, DEC, 1>(a, b, half_of(g.s, 4 * h + 1));
        v[4 * h + 2][i] = byte_pair_dequant<BF16, DEC, 2>(a, b, half_of(g.s, 4 * h + 2));
        v[4 * h + 3][i] = byte_pair_dequant<BF16, DEC, 3>(a, b, half_of(g.s, 4 * h + 3));
      }
  }
  // wide_b_offset<256>(8 rb, 8 cb + c) = base + 16 (c ^ fw)
  __device__ static uint8_t* base_of(uint8_t* Bs, int cb, int rb) {
    return Bs + wide_b_offset<256>(8 * rb, 8 * cb) - wide_slot(8 * cb) * 16 + cb * 128;
  }
  template <bool FAST>
  __device__ void store_all(const Raw& r, const Grp& g, uint8_t* Bs, int t) const {
    const int cb = cb_of(t), rb = rb_of(t);
    uint8_t* base = base_of(Bs, cb, rb);
    const int fw = (cb ^ (cb >> 3)) & 7;
    uint32_t v[8][2];
    dequant<2>(r, g, v);
#pragma unroll
    for (int c = 0; c < 8; ++c)
      *reinterpret_cast<kbh_u32x2*>(base + ((c ^ fw) << 4)) = kbh_u32x2{v[c][0], v[c][1]};
  }
  template <bool FAST>
  __device__ void store_half(const RawHalf& r, const Grp& g, uint8_t* Bs, int t, int half) const {
    const int cb = cb_of(t), rb = rb_of(t);
    uint8_t* base = base_of(Bs, cb, rb) + 4 * half;
    const int fw = (cb ^ (cb >> 3)) & 7;
    uint32_t v[8][1];
    dequant<1>(r, g, v);
#pragma unroll
    for (int c = 0; c < 8; ++c) *reinterpret_cast<uint32_t*>(base + ((c ^ fw) << 4)) = v[c][0];
  }
};

constexpr int kByteTiledMinM = 128;
constexpr int kByteWideMinM = 17;
constexpr int kByteWidePD = 4;

struct BytePlan {
  int spw, waves, ntiles, mb, mblocks, splits;
};

// Row blocks per wave (MB: 1 up to 16 rows, 2 up to 32, 4 up to 64, then 16-row blocks of 4),
// 4-step (128-deep) wave K ranges when they divide K (2 at MB = 4, for registers), waves per
// workgroup and K splits as for the W4 decode kernel.
bool plan_byte_decode(int M, int N, int K, BytePlan* p) {
  const int nsteps = K / 32;
  const int m16 = (M + 15) / 16;
  p->mb = m16 <= 1 ? 1 : (m16 <= 2 ? 2 : 4);
  const int smax = p->mb == 4 ? 2 : 4;
  p->spw = (nsteps % smax == 0) ? smax : (nsteps % 2 == 0 ? 2 : 1);
  p->ntiles = N / 128;
  p->mblocks = (m16 + p->mb - 1) / p->mb;
  p->splits = 0;
  p->waves = splitk_pick_waves(nsteps / p->spw, p->ntiles * p->mblocks, &p->splits);
  return p->waves > 0;
}

// K splits of the streaming kernel, or 0 where the decode kernel stays: it does while its grid is
// resident at once (two workgroups per CU), and where its estimated time is lower. Both estimates (us)
// are least-squares fits: the decode kernel's to 434 calls of 1 to 16 rows past 512 workgroups (4.6% rms),
// the streaming kernel's to 790 split counts of 54 layers (K from 2048 to 29568, N from 2560 to 65536; 7.6%
// rms; its rounds are of one workgroup per CU, and rows of a multiple of 1 KB cost it more: N=10240 is
// slower at every split). The 2.7% is about the smallest margin with which none of the 74 calls of M=1 and
// 16 among those came out more than 4% slower than on the decode kernel. (One rate and a constant for each
// kernel had chosen 22 of them 5 to 34% slower: 8192 x 10240 M=1 21.9 -> 26.7 us, 14336 x 10240 31.4 -> 42.0.)
inline int plan_byte_stream(int M, int N, int K, const BytePlan& d) {
  const long grid = (long)d.ntiles * d.splits;
  if (M > 16 || grid <= 512 || K % kByteStreamChunk != 0 || (size_t)K * N >= ((size_t)1 << 31)) return 0;
  const float mb = (float)K * N * 1e-6f, slice = (float)M * N * 8e-6f;  // MB of weights; of one split's slices
  float best = 0.973f * (6.89f + 0.149f * mb + (d.splits > 1 ? 0.28f * d.splits * slice : 0.f) +
                         1.02f * (float)((grid + 511) / 512) + (d.waves < 8 ? 0.33f : 0.f) + 0.0158f * M);
  const float fixed = 6.67f + (N % 1024 == 0 ? 0.0787f : 0.0637f) * mb + 0.0593f * M;
  int best_s = 0;
  // about one to at most the three workgroups a CU holds, at least two chunks per wave of a split K
  for (int s = 1; (long)d.ntiles * s <= 768; ++s) {
    if (s > 1 && K / kByteStreamChunk < 2 * kByteStreamWaves * s) break;
    const long wgs = (long)d.ntiles * s;
    if (wgs < 190) continue;
    const float row = wgs <= 256 ? 3.54e-3f : 3.37e-3f;  // of K and round
    const float t = fixed + row * (float)((wgs + 255) / 256) * ((float)K / s) + (s > 1 ? 0.196f * s * slice : 0.f);
    if (t < best) {
      best = t;
      best_s = s;
    }
  }
  return best_s;
}

struct ByteWide {
  WidePlan plan;
  int spg;
};

// Whether the decode kernel keeps a call of 17 to 127 rows from the wide tiles. It does while its
// grid is resident at once, so that every weight is in flight and few split-K slices are written:
// its blocks of 32 and 64 rows hold 116 to 228 registers, which leaves 8 waves to a CU. Workgroups of
// under three waves have too little in flight each (K=N=1024 M=65 17.0 against 12.0 us), and above
// one workgroup per CU up to 64 rows it also takes whole multiples of 8 workgroups (xcd_remap and the
// slice sum placed by it: 3072 x 3712 M=64 19.6 against 16.1, 3072 x 3072 15.4 / 15.7). From 65 rows
// the second row block of a little over one round is mostly padding that costs no MFMAs
// (2560 x 4096 M=72 13.9 against 18.4). Measured over 169 layers of K and N from 1024 to 14336 and 208
// with N of 128 mod 256: the choice is 0.3% from the faster kernel on average and never more than 11%
// slower than decode, where "up to 64 rows and one workgroup per CU" lost up to 46% (M=127: 4096 x 2048
// 13.8 against 20.0, 2048 x 4096 14.0 / 19.9; M=17: 4096 x 6144 13.1 / 14.1).
// The int8 base of the multi-LoRA linear from 33 rows (`int8`): only one workgroup per CU, or full ones whose second
// row block is mostly padding. Beyond that int8 codes cost the decode kernel more and the wide tiles less than FP8
// codes do (the GEMM alone, 3584 x 3584 and 64 rows: 16.4 against 12.1 us, FP8 15.2 / 13.4), and the slice sum that
// the decode plan makes faster (FP8 3.9 / 4.3) is replaced by this linear's last kernel.
// Of 364 calls (28 layers, 17 to 127 rows, fp16) 25 were more than 4% slower than on the wide tiles under the
// line of the FP8 weights (3584 x 3584 r=8 T=57 19.9 against 23.3 us, 2560 x 2560 T=96 22.7 / 25.3) and none is now.
inline bool byte_decode_stays(int M, const BytePlan& d, bool int8) {
  const int grid = d.ntiles * d.splits * d.mblocks;
  if (int8 && M > 32 && grid > 256 && !(M > 64 && d.waves == 8)) return false;
  const bool resident = grid <= 256 * (d.waves < 8 ? 8 / d.waves : 1);
  if (M <= 64) return grid <= 256 || (resident && d.waves >= 4 && grid % 8 == 0);
  return (resident && d.waves >= 3) || (M <= 96 && d.waves >= 5 && grid <= 320);
}

// Wide tiles from kByteWideMinM rows: the W4A16 geometry (64-row tiles up to 64 rows, 128-row
// ones up to 128, then 128 or 256 rows by the estimate). They replace
// tiled_f16_gemm's 256 x 128 tiles, which split no K (K=14336 N=4096: 32 workgroups and ~300 us
// at every M from 128 to 1024; now 30.7 / 43.0 / 75.2 / 124 us at M=128 / 256 / 512 / 1024, and
// 342 -> 226 at 2048), and the decode kernel's 32- and 64-row blocks where those take several rounds
// (M=32 26.2 -> 19.4, M=48 42.9 -> 21.4, M=96 73.2 -> 28.4; 8192 x 28672 M=32 85.5 -> 66.9).
bool plan_byte_wide(int M, int N, int K, int block, bool int8, ByteWide* w) {
  if (M < kByteWideMinM || N < 256) return false;
  // the kernels stage x with 32-bit offsets
  if ((size_t)(M + 256) * K * 2 >= ((size_t)1 << 31)) return false;
  BytePlan d;
  if (M < kByteTiledMinM && plan_byte_decode(M, N, K, &d) && byte_decode_stays(M, d, int8)) return false;
  w->spg = block / 32;
  const int unit = wide_iteration(w->spg, kByteWidePD) / 2;
  return plan_wide(M, N, K, 256, 32, unit, unit, 256, kHalfCosts, &w->plan, M <= 64 ? 64 : 128);
}

template <bool BF16, int DEC, int SPG>
void launch_byte_wide(const ByteWide& w, const void* x, const void* wt, const void* scales, void* y,
                      float* slices, int M, int N, int K, int block, hipStream_t st) {
  using E = WideHalf<BF16>;
  using BP = ByteWidePolicy<BF16, DEC>;
  using EP = HalfOut<BF16>;
  const BP bp{(const uint8_t*)wt, (const uint16_t*)scales, N, block};
  const EP ep{(uint16_t*)y, N};
  const WidePlan& p = w.plan;
  if (p.tm == 256)
    hipLaunchKernelGGL((tiled_ws256_gemm<E, SPG, BP, EP, kByteWidePD>), dim3(p.grid), dim3(768), 0,
                       st, x, bp, ep, slices, M, N, K, p.sp);
  else if (p.tm == 128)  // bf16's fp32 dequantization: two producer sets (M=256 44.4 -> 43.6 us)
    hipLaunchKernelGGL((tiled_ws_gemm<E, 128, 2, SPG, BP, EP, DenseRows, kByteWidePD, BF16 ? 2 : 1, true>),
                       dim3(p.grid), dim3(BF16 ? 768 : 512), 0, st, x, bp, ep, slices, M, N, K, p.sp, DenseRows{M});
  else
    hipLaunchKernelGGL((tiled_ws_gemm<E, 64, 2, SPG, BP, EP, DenseRows, kByteWidePD, 2>),
                       dim3(p.grid), dim3(768), 0, st, x, bp, ep, slices, M, N, K, p.sp, DenseRows{M});
}

// The decode kernel's plan when byte_gemm_run takes that kernel for this shape.
bool byte_takes_decode(int M, int N, int K, int block, bool int8, BytePlan* p) {
  ByteWide w;
  if (plan_byte_wide(M, N, K, block, int8, &w)) return false;
  if (M >= kByteTiledMinM && K % (TBK * TDEPTH) == 0) return false;
  return plan_byte_decode(M, N, K, p);
}

// Runs the GEMM; with `defer_sum` and a split K the slices are left in the workspace
// (acc[splits][M][N] fp32) for the caller to sum, and *splits_out tells how many (1: y written).
// `side` runs with the decode kernel's launch; where another kernel runs, the caller launches it.
template <bool BF16, int DEC, class SIDE = NoSide>
int byte_gemm_run(const void* x, const void* w, const void* scales, void* y, void* workspace,
                  size_t workspace_bytes, int M, int N, int K, int block, hipStream_t st,
                  bool defer_sum = false, int* splits_out = nullptr, SIDE side = SIDE{}) {
  if (splits_out) *splits_out = 1;
  ByteWide wide;
  bool is_wide = plan_byte_wide(M, N, K, block, DEC == kDecInt8, &wide);
  if (is_wide) {  // without room for the slices, the kernels that ran the call before the wide tiles
    const size_t need = wide_workspace_bytes(M, N, wide.plan.splits);
    is_wide = need == 0 || (workspace && workspace_bytes >= need);
  }
  if (is_wide) {
    const int splits = wide.plan.splits;
    if (splits > 1 && !aligned16(workspace)) return KBH_ERR_ALIGN;
    float* slices = (float*)workspace;
    switch (wide.spg) {
      case 1: launch_byte_wide<BF16, DEC, 1>(wide, x, w, scales, y, slices, M, N, K, block, st); break;
      case 2: launch_byte_wide<BF16, DEC, 2>(wide, x, w, scales, y, slices, M, N, K, block, st); break;
      case 4: launch_byte_wide<BF16, DEC, 4>(wide, x, w, scales, y, slices, M, N, K, block, st); break;
      default: launch_byte_wide<BF16, DEC, 8>(wide, x, w, scales, y, slices, M, N, K, block, st); break;
    }
    if (splits_out) *splits_out = splits;
    if (splits > 1 && !defer_sum) {
      using EP = HalfOut<BF16>;
      const size_t n4 = (size_t)M * N / 4;
      hipLaunchKernelGGL((wide_reduce_kernel<WideHalf<BF16>, EP>), dim3((unsigned)((n4 + 255) / 256)),
                         dim3(256), 0, st, slices, EP{(uint16_t*)y, N}, N, n4, splits);
    }
    return launch_status();
  }
  if (M >= kByteTiledMinM && K % (TBK * TDEPTH) == 0) {
    const ByteSlabPolicy<BF16, DEC> bp{(const uint8_t*)w, (const uint16_t*)scales, N, block};
    hipLaunchKernelGGL((tiled_f16_gemm<BF16, ByteSlabPolicy<BF16, DEC>>), tiled_f16_grid(M, N),
                       dim3(256), 0, st, (const uint16_t*)x, bp, (uint16_t*)y, M, N, K);
    return launch_status();
  }
  BytePlan pl;
  if (!plan_byte_decode(M, N, K, &pl)) return KBH_ERR_SHAPE;
  if constexpr (DEC == kDecE4M3 && !SIDE::kAny) {
    if (const int s = plan_byte_stream(M, N, K, pl)) {
      const size_t need = splitk_workspace_bytes(M, N, s);
      if (need > 0 && (!workspace || workspace_bytes < need)) return KBH_ERR_WORKSPACE;
      if (need > 0 && !aligned16(workspace)) return KBH_ERR_ALIGN;
      hipLaunchKernelGGL((byte_stream_kernel<BF16>), dim3(pl.ntiles * s), dim3(64 * kByteStreamWaves),
                         0, st, (const uint16_t*)x, (const uint8_t*)w, (const uint16_t*)scales,
                         (uint16_t*)y, (float*)workspace, M, N, K, block, s);
      if (splits_out) *splits_out = s;
      if (s > 1 && !defer_sum)
        launch_splitk_sum(reinterpret_cast<const kbh_f32x4*>(workspace), HalfOut<BF16>{(uint16_t*)y, N},
                          M, N, pl.ntiles, 128, s, st);
      return launch_status();
    }
  }
  const int spw = pl.spw, waves = pl.waves, splits = pl.splits;
  const size_t need = splitk_workspace_bytes(M, N, splits);
  if (need > 0 && (!workspace || workspace_bytes < need)) return KBH_ERR_WORKSPACE;
  if (need > 0 && !aligned16(workspace)) return KBH_ERR_ALIGN;
  dim3 grid(pl.ntiles * splits + side.blocks, pl.mblocks);
  float* acc = (float*)workspace;
#define KBH_BYTE_DEC(SPW_, MB_)                                                                  \
  if (spw == SPW_ && pl.mb == MB_)                                                               \
    hipLaunchKernelGGL((byte_decode_kernel<SPW_, BF16, DEC, MB_, SIDE>), grid, dim3(waves * 64), \
                       0, st, (const uint16_t*)x, (const uint8_t*)w, (const uint16_t*)scales,    \
                       (uint16_t*)y, acc, M, N, K, block, splits, side);
  KBH_BYTE_DEC(4, 1) else KBH_BYTE_DEC(2, 1) else KBH_BYTE_DEC(1, 1)
  else KBH_BYTE_DEC(4, 2) else KBH_BYTE_DEC(2, 2) else KBH_BYTE_DEC(1, 2)
  else KBH_BYTE_DEC(2, 4) else KBH_BYTE_DEC(1, 4)
#undef KBH_BYTE_DEC
  if (splits_out) *splits_out = splits;
  if (splits > 1 && !defer_sum)
    launch_splitk_sum(reinterpret_cast<const kbh_f32x4*>(acc), HalfOut<BF16>{(uint16_t*)y, N}, M, N,
                      pl.ntiles, 128, splits, st);
  return launch_status();
}

// Workspace bytes of byte_gemm_run for this shape (0 when K is not split).
size_t byte_gemm_workspace_bytes(int M, int N, int K, int block, bool int8) {
  if (M < 1 || N < 128 || K < 32 || block < 32 || K % block != 0) return 0;
  ByteWide w;
  if (plan_byte_wide(M, N, K, block, int8, &w)) return wide_workspace_bytes(M, N, w.plan.splits);
  if (M >= kByteTiledMinM && K % (TBK * TDEPTH) == 0) return 0;  // tiled path: no split
  BytePlan p;
  if (!plan_byte_decode(M, N, K, &p)) return 0;
  const int s = plan_byte_stream(M, N, K, p);  // FP8 weights; the int8 base takes the decode plan
  const size_t dec = splitk_workspace_bytes(M, N, p.splits), str = splitk_workspace_bytes(M, N, s);
  return dec > str ? dec : str;
}

}  // namespace
}  // namespace kbh
