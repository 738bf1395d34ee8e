// Few-row tile of the dense GEMMs: C = A . B^T on v_mfma_f32_16x16x4_f32 with K
// split over the waves of a block.
#pragma once

#include "gpu_common.h"
#include "mfma_tile.h"

namespace moe {

// A block of NW waves computes RM x RN blocks of 16x16, each wave all of them
// over its own slice of K, NS - 1 pieces of 32 k ahead in registers, and no
// barrier until the waves' sums meet in LDS.  Few rows leave few tiles, so a
// tile that one CU works through from end to end takes as long as the whole
// product: splitting K over a block's waves keeps many loads in flight and
// small tiles keep every CU busy.  Loads follow the memory (8 lanes read the
// 128 bytes of a row's piece): the MFMA's operand layout, whose neighbouring
// lanes hold different rows, loads one lane's 16 bytes per cycle (37 B/ns per
// CU measured, 4x below contiguous lanes).  The pieces pass through a
// wave-private LDS buffer into the operand layout, 16-byte chunk c of row r at
// c ^ (r % 8).  The products are in transposed form (B rows as the first
// operand), so a lane's four results are consecutive columns.  fp32 MFMAs: with
// tiles this small, splitting into bf16 parts (split_tile.h) costs what it saves.
// Measured, M x N x K: 1 x 2048 x 2048 34 (64x128 fp32 tiles) -> 5.9 us (2.9
// TB/s), 9 x 6144 x 2048 35 -> 12.4 (4.1 TB/s), 100 x 2048 x 2048 74 -> 13.7
// (61 TFLOP/s): bound by the launch and the loads' latency, HBM, and the fp32
// MFMAs of an uneven number of tiles per CU.
template <int RM_, int RN_, int NW_, int NS_, int CH_ = 1> struct SkinnyTile {
  static constexpr int RM = RM_, RN = RN_, NW = NW_, NS = NS_;
  static constexpr int CH = CH_;  // chains of rounded additions a wave's sum is cut into (1, 2, 4)
  static constexpr int BM = RM * 16, BN = RN * 16, PITCH = BN + 4;
  static constexpr int STAGE = (BM + BN) * 32;  // floats of a wave's LDS buffer
  static constexpr int RED = BM * PITCH;        // floats of a wave's sums
  static constexpr size_t LDS_BYTES = (size_t)NW * (STAGE > RED ? STAGE : RED) * sizeof(float);
  static_assert(LDS_BYTES <= 65536, "no LDS attribute needed");
};

// The waves' sums of one tile, left in LDS after a barrier: rows m0 .. of A
// [M][32 np] (rows past M are zero) times the tile's B rows, row r at float
// brow(r) of the piece's base bsrc(p, k0) (k0: the piece's first column there;
// every row within bbytes of the base).
template <typename CF, typename BRow, typename BSrc>
__device__ __forceinline__ void skinny_tile(float *lds, const float *A, int M, int m0, int np,
                                            uint32_t bbytes, BRow brow, BSrc bsrc) {
  constexpr int RM = CF::RM, RN = CF::RN, NW = CF::NW, NS = CF::NS, CH = CF::CH;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lq = lane >> 4;
  const int K = np * 32;
  const __amdgpu_buffer_rsrc_t ar = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float *>(A), 0, (int)((uint32_t)M * K * 4u), kBufferRsrcWord3);
  // lane l of a load: row l / 8 of 8, 16-byte chunk l % 8
  const int ll = lane >> 3, lc = lane & 7;
  uint32_t aoff[2 * RM], boff[2 * RN];
#pragma unroll
  for (int i = 0; i < 2 * RM; ++i) {
    const int row = m0 + 8 * i + ll;
    aoff[i] = row < M ? (uint32_t)(row * K + 4 * lc) * 4u : kTileOOB;
  }
#pragma unroll
  for (int i = 0; i < 2 * RN; ++i) boff[i] = (uint32_t)(brow(8 * i + ll) + 4 * lc) * 4u;

  // this wave's pieces: [p0, p1).  Pieces past the end come through empty
  // descriptors (zeros, no traffic), so every load is unconditional and the
  // compiler's count of loads in flight stays exact.
  const int per = (np + NW - 1) / NW;
  const int p0 = min(wave * per, np), p1 = min(p0 + per, np);
  f32x4 sa[NS][2 * RM], sb[NS][2 * RN];
  auto load = [&](int p, int set) {
    const bool in = p < p1;
    int k0 = 0;
    const float *bp = bsrc(in ? p : 0, k0);
    const __amdgpu_buffer_rsrc_t br = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(bp), 0, in ? (int)bbytes : 0, kBufferRsrcWord3);
    const __amdgpu_buffer_rsrc_t arp = in ? ar : br;
    const int aks = in ? p * 128 : 0, bks = k0 * 4;
#pragma unroll
    for (int i = 0; i < 2 * RN; ++i)
      sb[set][i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(br, boff[i], bks, 0));
#pragma unroll
    for (int i = 0; i < 2 * RM; ++i)
      sa[set][i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(arp, aoff[i], aks, 0));
  };
  // the wave's buffer: B rows, then A rows, of 32 floats
  float *stage = lds + (size_t)wave * CF::STAGE;
  float *wr = stage + ll * 32 + (lc ^ ll) * 4;
  const float *rd = stage + lr * 32;
  const int rc[2] = {(lq ^ (lr & 7)) * 4, ((lq + 4) ^ (lr & 7)) * 4};
  f32x4 acc[CH][RM][RN];
#pragma unroll
  for (int c = 0; c < CH; ++c)
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
      for (int j = 0; j < RN; ++j) acc[c][i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int s = 0; s < NS - 1; ++s) {
    load(p0 + s, s);
    // in the loop's order: mixed, its first wait would be for all of them
    __builtin_amdgcn_sched_barrier(0);
  }
  for (int p = p0; p < p1; p += NS) {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      load(p + s + NS - 1, (s + NS - 1) % NS);
      __builtin_amdgcn_sched_barrier(0);
      // a wave's LDS operations complete in order: no wait between the writes
      // and the reads, and none before the next piece's writes
#pragma unroll
      for (int i = 0; i < 2 * RN; ++i) st4(wr + i * 256, sb[s][i]);
#pragma unroll
      for (int i = 0; i < 2 * RM; ++i) st4(wr + (RN * 2 + i) * 256, sa[s][i]);
      __builtin_amdgcn_wave_barrier();
      f32x4 af[RM][2], bf[RN][2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int j = 0; j < RN; ++j) bf[j][h] = ld4(rd + j * 512 + rc[h]);
#pragma unroll
        for (int i = 0; i < RM; ++i) af[i][h] = ld4(rd + (RN + i) * 512 + rc[h]);
      }
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int i = 0; i < RM; ++i)
#pragma unroll
            for (int j = 0; j < RN; ++j)
              acc[(h + 2 * q) % CH][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                  bf[j][h][q], af[i][h][q], acc[(h + 2 * q) % CH][i][j], 0, 0, 0);
    }
  }

#pragma unroll
  for (int c = 1; c < CH; ++c)
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
      for (int j = 0; j < RN; ++j) acc[0][i][j] += acc[c][i][j];
  __syncthreads();  // every wave is done with its buffer
  // lane l of a block: row l % 16, columns 4 (l / 16) .. + 3
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < RN; ++j)
      st4(lds + (size_t)(wave * CF::BM + 16 * i + lr) * CF::PITCH + 16 * j + 4 * lq, acc[0][i][j]);
  __syncthreads();
}

// Four columns from col (a multiple of 4) of a row of the tile, over the waves
// in order.
template <typename CF>
__device__ __forceinline__ f32x4 skinny_sum(const float *lds, int row, int col) {
  f32x4 v = ld4(lds + (size_t)row * CF::PITCH + col);
#pragma unroll
  for (int w = 1; w < CF::NW; ++w) v += ld4(lds + (size_t)(w * CF::BM + row) * CF::PITCH + col);
  return v;
}

}  // namespace moe
