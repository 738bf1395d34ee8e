// Split-bf16 tile of the dense and grouped GEMMs: C = A . B^T for fp32 A and B
// on v_mfma_f32_32x32x16_bf16.
//
// The fp32 matrix instruction peaks at 157 TFLOP/s on this chip, the bf16 one
// at 2.5 PFLOP/s.  Every fp32 value of at least 2^-110 is exactly the sum of
// three bf16 values (8 significand bits each, rounded to nearest, so each part
// is at most 2^-8 of the one before), and a product of two values is then nine
// bf16 products, of which six are taken,
//   a2 b0 + a0 b2 + a1 b1 + a1 b0 + a0 b1 + a0 b0.
// The other three are together at most 2^-24 of the product (2^-28 on
// average), as much as the rounding of one fp32 product: an output that is a
// single product is within 1 ulp, where the fp32 instruction's is within half.
// The six are exact in fp32 and accumulate in fp32, 16 k per instruction, so a
// sum of K products takes 6 K / 16 roundings where the fp32 instruction takes
// K / 2: measured against 64-bit sums its error is smaller (K = 2048 7.0e-7,
// 8.1e-7).  Six of them take 192 cycles per 32x32x16 block where fp32 takes 512.
//
// Values the split cannot carry leave outputs that a wave computes again with
// the fp32 instruction: infinities, NaN and magnitudes above the largest bf16
// (which round to infinity) a NaN or an infinity in every output they reach, as
// does an fp32 overflow; magnitudes below about 2^-110, whose lowest parts fall
// under bf16's smallest subnormal, 2^-133, an output too small for its operands
// (kSplitFloor).  The wave takes those outputs alone from its second pass, so
// that no row's bits depend on what other rows of its tile hold.
#pragma once

#include "gpu_common.h"
#include "mfma_tile.h"

namespace moe {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// x, y -> the packed bf16 pairs of their three parts (11 VALU operations; with
// integer rounding and byte permutes instead of conversions as fast).
__device__ __forceinline__ void split_pair(float x, float y, uint32_t &p0, uint32_t &p1, uint32_t &p2) {
  p0 = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{x, y}, bf16x2));
  x -= __builtin_bit_cast(float, p0 << 16);
  y -= __builtin_bit_cast(float, p0 & 0xFFFF0000u);
  p1 = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{x, y}, bf16x2));
  x -= __builtin_bit_cast(float, p1 << 16);
  y -= __builtin_bit_cast(float, p1 & 0xFFFF0000u);
  p2 = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{x, y}, bf16x2));
}

// Eight floats, as two float4s, to the three parts' operand registers.
__device__ __forceinline__ void split8(const f32x4 (&v)[2], bf16x8 (&out)[3]) {
  u32x4 p[3];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    uint32_t p0, p1, p2;
    split_pair(v[j >> 1][(j & 1) * 2], v[j >> 1][(j & 1) * 2 + 1], p0, p1, p2);
    p[0][j] = p0;
    p[1][j] = p1;
    p[2][j] = p2;
  }
#pragma unroll
  for (int q = 0; q < 3; ++q) out[q] = __builtin_bit_cast(bf16x8, p[q]);
}

// The sum of a value's parts is off by at most 2^-134 (the instruction and the
// conversion keep subnormals), so an output by K 2^-134 (|a| + |b|), |a| and |b|
// the largest magnitudes of its row and its column: at most 2^-25 of an output
// of kSplitFloor K (|a| + |b|), below which it is computed again.  The maxima
// take half an instruction per value in the staging, where the split takes 5.5.
constexpr float kSplitFloor = 0x1p-109f;

// The six products in ascending size, as (part of A, part of B).
constexpr int kSplitProducts = 6;
__device__ constexpr int kSplitA[kSplitProducts] = {2, 0, 1, 1, 0, 0};
__device__ constexpr int kSplitB[kSplitProducts] = {0, 2, 1, 0, 1, 0};

// max(m, |x|, |y|) in one instruction; a NaN makes it a NaN.
__device__ __forceinline__ float max_abs(float m, float x, float y) {
  return __builtin_elementwise_maximum(__builtin_elementwise_maximum(m, fabsf(x)), fabsf(y));
}

// v of another lane of the quad.
template <int CTRL> __device__ __forceinline__ float quad_perm(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}

// Tile of BM rows x BN columns, each of the four waves AM x 2 blocks of 32x32
// (BN = 128: 2 x 2 waves, BN = 64: 4 x 1).  Slabs of 32 k: thread t stages 8
// floats of rows t / 4 + 64 i (two float4s, 16 k apart, so four threads read
// 64 contiguous bytes), splits them and writes one 16-byte chunk per plane;
// both operands permute k alike.
// Neighbouring lanes must hold neighbouring addresses: a load whose lanes hold
// different rows moves 16 bytes per cycle, not 64.  LDS holds [3 planes][rows][4 chunks], chunk
// c of row r at c ^ swizzle(r), so the 16-byte reads of neighbouring rows fall
// in different banks without padding (no conflicts counted) and several blocks
// share a CU: one splits its next slab while another's MFMAs run.
template <int BM_, int BN_, int NBUF_ = 1> struct SplitTile {
  static constexpr int BM = BM_, BN = BN_, BK = 32;
  // LDS slab buffers and slabs of global loads in flight.  One: two barriers
  // per slab, the other blocks of the CU fill the waits (three blocks at 128
  // rows).  Two: the next slab is split between the MFMAs of this one, one
  // barrier per slab; faster where only two blocks fit anyway (64-row expert
  // units, 512 tokens: 522 -> 495 us), slower where it costs a block (64-row
  // dense tiles at M=2664 N=2048: 140 -> 155 us).
  static constexpr int NBUF = NBUF_, NS = NBUF;
  static constexpr int WAVES_N = BN / 64, WAVES_M = kThreads / 64 / WAVES_N;
  static constexpr int AM = BM / 32 / WAVES_M;  // 32-row blocks per wave
  static constexpr int A_PASSES = BM / 64, PASSES = (BM + BN) / 64;  // float4 pairs per thread and slab
  static constexpr int PLANE = (BM + BN) * BK;  // bf16 values per plane
  static constexpr size_t LDS_BYTES = (size_t)3 * PLANE * 2 * NBUF;
  static constexpr int LDS_FLOATS = (int)(LDS_BYTES / sizeof(float));
  static_assert(BM % 64 == 0 && (BN == 64 || BN == 128) && AM * WAVES_M * 32 == BM, "whole row blocks");
};

__device__ __forceinline__ int split_swizzle(int r) { return ((r >> 1) & 3) ^ ((r >> 3) & 1); }

// Arguments as mfma_tile's (mfma_tile.h); out.store1(byte offset, value)
// stores one float.  GATED: B rows come in groups of 32 of W1 and 32 of W3, a
// wave's two column blocks, and silu(W1 x) * (W3 x) is stored.
template <typename TL, bool GATED, typename Out, typename Ready = NoWait, typename Claim = int *>
__device__ __forceinline__ int split_tile(float *lds, const float *abase, uint32_t abytes,
                                          const int *aoff, int rows_valid, const float *brow0, int K,
                                          const Out &out, int row0, int ldo, int col0, Claim head,
                                          Ready ready = Ready{}) {
  constexpr int AM = TL::AM, BM = TL::BM, PA = TL::A_PASSES, PASSES = TL::PASSES;
  uint16_t *planes = reinterpret_cast<uint16_t *>(lds);
  // through asm, so that the compiler cannot compute a tile's offsets outside
  // the caller's task loop: every kind of tile's, held throughout, took the
  // registers of the third block per CU
  int tid = threadIdx.x;
  asm("" : "+v"(tid));
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const __amdgpu_buffer_rsrc_t ar =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(abase), 0, (int)abytes, kBufferRsrcWord3);
  const __amdgpu_buffer_rsrc_t br = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float *>(brow0), 0, (int)((uint32_t)TL::BN * K * 4u), kBufferRsrcWord3);

  // staging: row lrow + 64 i (A rows, then B rows), float4s lq and lq + 4
  const int lrow = tid >> 2, lq = tid & 3;
  uint32_t a_src[PA];
#pragma unroll
  for (int i = 0; i < PA; ++i) {
    const int r = lrow + 64 * i;
    a_src[i] = r < rows_valid ? (uint32_t)(aoff[r] + lq * 4) * 4u : kTileOOB;
  }
  const uint32_t b_src = (uint32_t)(lrow * K + lq * 4) * 4u;
  // slabs past the end come through empty descriptors: zeros, no traffic, and
  // the compiler's count of loads in flight stays exact across the loop
  const __amdgpu_buffer_rsrc_t none =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(brow0), 0, 0, kBufferRsrcWord3);
  const int nslab = K / TL::BK;
  constexpr int NS = TL::NS;
  f32x4 st[NS][PASSES][2];
  auto load = [&](int slab, int set) {
    const bool in = slab < nslab;
    const __amdgpu_buffer_rsrc_t arp = in ? ar : none, brp = in ? br : none;
    const int ks = in ? slab * TL::BK * 4 : 0;
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
      // what is the same for all lanes in the scalar offset where registers
      // decide the blocks per CU; two buffers have registers to spare and are
      // faster with it in the vector offset (520 tokens 496 / 502 us)
      const uint32_t uni = i < PA ? 0u : (uint32_t)((i - PA) * 64) * (uint32_t)K * 4u;
      const uint32_t own = i < PA ? a_src[i < PA ? i : 0] : b_src;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const uint32_t so = uni + 64 * h;
        st[set][i][h] = __builtin_bit_cast(
            f32x4, __builtin_amdgcn_raw_buffer_load_b128(i < PA ? arp : brp, TL::NBUF == 1 ? own : own + so,
                                                         TL::NBUF == 1 ? (int)(ks + so) : ks, 0));
      }
    }
  };
  // (lrow + 64 i) * 32 keeps lrow's swizzle: 64 i changes neither of its bits
  uint16_t *wr = planes + lrow * TL::BK + (lq ^ split_swizzle(lrow)) * 8;
  float mag[PASSES];  // largest magnitude this thread staged of each of its rows
#pragma unroll
  for (int i = 0; i < PASSES; ++i) mag[i] = 0.0f;
  auto track = [&](int set, int i) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      mag[i] = max_abs(mag[i], st[set][i][h][0], st[set][i][h][1]);
      mag[i] = max_abs(mag[i], st[set][i][h][2], st[set][i][h][3]);
    }
  };
  auto store = [&](int set, int buf) {
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
      if constexpr (TL::NBUF == 1) track(set, i);
      bf16x8 p[3];
      split8(st[set][i], p);
#pragma unroll
      for (int q = 0; q < 3; ++q)
        *reinterpret_cast<bf16x8 *>(wr + (3 * buf + q) * TL::PLANE + i * 64 * TL::BK) = p[q];
    }
  };
  // two buffers: a set's values stay until the next step's loads
  auto track_late = [&](int set) {
#pragma unroll
    for (int i = 0; i < PASSES; ++i) track(set, i);
  };

  // fragments: lane l supplies row l % 32, chunk 2 kk + l / 32 of a slab
  const int wm = wave % TL::WAVES_M, wn = wave / TL::WAVES_M;
  const int lr = lane & 31, lh = lane >> 5;
  const int sw = split_swizzle(lr);  // row blocks are 32 rows apart: the same swizzle
  const uint16_t *a_rd = planes + (wm * AM * 32 + lr) * TL::BK;
  const uint16_t *b_rd = planes + (BM + wn * 64 + lr) * TL::BK;
  floatx16 acc[AM][2];
#pragma unroll
  for (int i = 0; i < AM; ++i)
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][c][r] = 0.0f;

  if constexpr (Ready::kActive) {
    if (wave == 0)
      for (int j = 0; j < NS; ++j) ready.wait(j);
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    load(j, j);
    __builtin_amdgcn_sched_barrier(0);  // in the loop's order: see the waits in it
  }
  // The MFMAs go before other waves' instructions: those of the wave that
  // splits beside them then fill the cycles between, which pays for the maxima
  // (4096 tokens 2030 -> 1997 us).
  auto compute = [&](int kk, int buf) {
    const int co = ((2 * kk + lh) ^ sw) * 8 + 3 * buf * TL::PLANE;
    bf16x8 bf[2][3];
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int p = 0; p < 3; ++p)
        bf[c][p] = *reinterpret_cast<const bf16x8 *>(b_rd + p * TL::PLANE + c * 32 * TL::BK + co);
#pragma unroll
    for (int i = 0; i < AM; ++i) {
      bf16x8 af[3];
#pragma unroll
      for (int p = 0; p < 3; ++p)
        af[p] = *reinterpret_cast<const bf16x8 *>(a_rd + p * TL::PLANE + i * 32 * TL::BK + co);
#pragma unroll
      for (int m = 0; m < kSplitProducts; ++m)
#pragma unroll
        for (int c = 0; c < 2; ++c)
          acc[i][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[kSplitA[m]], bf[c][kSplitB[m]],
                                                              acc[i][c], 0, 0, 0);
    }
  };
  if constexpr (TL::NBUF == 1) {
    for (int t = 0; t < nslab; ++t) {
      store(0, 0);
      // the A columns of the slab loaded next, before the barrier
      if constexpr (Ready::kActive)
        if (wave == 0) ready.wait(t + 1);
      __syncthreads();
      load(t + 1, 0);
      __builtin_amdgcn_sched_barrier(0);  // not sunk among the MFMAs
      __builtin_amdgcn_s_setprio(1);
      compute(0, 0);
      compute(1, 0);
      __builtin_amdgcn_s_setprio(0);
      __syncthreads();
    }
  } else {
    store(0, 0);
    track_late(0);
    if constexpr (Ready::kActive)
      if (wave == 0) ready.wait(2);
    __syncthreads();
    for (int s = 0; s < nslab; s += 2) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int t = s + u;
        if (t >= nslab) break;
        load(t + 2, u);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(1);
        compute(0, u);
        store(1 - u, 1 - u);  // slab t + 1 (past the end: zeros into a buffer nobody reads)
        compute(1, u);
        track_late(1 - u);
        __builtin_amdgcn_s_setprio(0);
        if constexpr (Ready::kActive)
          if (wave == 0) ready.wait(t + 3);
        __syncthreads();
      }
    }
  }

  const int next = tid == 0 ? claim_next(head) : 0;

  int et = tid;  // and the epilogue's offsets not before the slab loop
  asm("" : "+v"(et));
  const int elr = et & 31, elh = (et >> 5) & 1;

  // The rows' magnitudes, in LDS (free after the last barrier): A rows, then
  // B rows, from the four threads that staged each (lanes ^ 1, ^ 2).
#pragma unroll
  for (int i = 0; i < PASSES; ++i) {
    mag[i] = __builtin_elementwise_maximum(mag[i], quad_perm<0xB1>(mag[i]));
    mag[i] = __builtin_elementwise_maximum(mag[i], quad_perm<0x4E>(mag[i]));
    // an output of a zero row or column is zero: no limit
    if ((et & 3) == 0)
      lds[(et >> 2) + 64 * i] = mag[i] != 0.0f ? mag[i] * ((float)K * kSplitFloor) : -__builtin_inff();
  }
  __syncthreads();

  // Elements the parts do not give: not finite, or below the limit of their
  // row and column (kSplitFloor).
  const float mb[2] = {lds[BM + wn * 64 + elr], lds[BM + wn * 64 + 32 + elr]};
  auto row_limit = [&](int i, int r) {
    return lds[wm * AM * 32 + i * 32 + 8 * (r >> 2) + 4 * elh + (r & 3)];
  };
#pragma unroll
  for (int i = 0; i < AM; ++i) {
    // a lane's smallest result above its row's limit against its column's
    float top = 0.0f, low[2] = {__builtin_inff(), __builtin_inff()};
#pragma unroll
    for (int r = 0; r < 16; r += 2)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const float x = acc[i][c][r], y = acc[i][c][r + 1];
        top = max_abs(top, x, y);
        low[c] = __builtin_elementwise_minimum(
            __builtin_elementwise_minimum(low[c], fabsf(x) - row_limit(i, r)), fabsf(y) - row_limit(i, r + 1));
      }
    if (__any(!(top <= __FLT_MAX__ && low[0] >= mb[0] && low[1] >= mb[1]))) {
      // fp32 MFMAs with operands straight from memory: lane l supplies row
      // l % 32 at k offset 4 (l / 32) of each 8-wide k group
      const int row = wm * AM * 32 + i * 32 + elr;
      const uint32_t ao = row < rows_valid ? (uint32_t)(aoff[row] + 4 * elh) * 4u : kTileOOB;
      const uint32_t bo = (uint32_t)((wn * 64 + elr) * K + 4 * elh) * 4u;
      floatx16 f[2];
#pragma unroll
      for (int r = 0; r < 16; ++r) f[0][r] = f[1][r] = 0.0f;
#pragma unroll 1
      for (int k = 0; k < K; k += 16) {
        f32x4 av[2], bv[2][2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          av[h] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(ar, ao, (k + 8 * h) * 4, 0));
#pragma unroll
          for (int c = 0; c < 2; ++c)
            bv[c][h] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                     br, bo + (uint32_t)(c * 32 * K) * 4u, (k + 8 * h) * 4, 0));
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int c = 0; c < 2; ++c)
              f[c] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[h][q], bv[c][h][q], f[c], 0, 0, 0);
      }
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (!(fabsf(acc[i][c][r]) - row_limit(i, r) >= mb[c] && fabsf(acc[i][c][r]) <= __FLT_MAX__))
            acc[i][c][r] = f[c][r];
    }
    // lane l holds column l % 32 and rows 8 (r / 4) + 4 (l / 32) + r % 4 of
    // each block, so a store writes 128 contiguous bytes of two rows
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = wm * AM * 32 + i * 32 + 8 * (r >> 2) + 4 * elh + (r & 3);
      if (row < rows_valid) {
        const size_t o = (size_t)(row0 + row) * ldo + col0;
        if (GATED) {
          out.store1((uint32_t)((o + wn * 32 + elr) * 4), silu(acc[i][0][r]) * acc[i][1][r]);
        } else {
          out.store1((uint32_t)((o + wn * 64 + elr) * 4), acc[i][0][r]);
          out.store1((uint32_t)((o + wn * 64 + 32 + elr) * 4), acc[i][1][r]);
        }
      }
    }
  }
  return next;
}

}  // namespace moe
