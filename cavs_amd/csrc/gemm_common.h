// What the matrix product kernels share: their arguments, how workgroups map to tiles, which part of
// K a tile runs over and how its accumulators are stored.
#pragma once
#include "common.h"

namespace cavs {

typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kThreads = 256;

struct GemmArgs {
  int M, N, K;
  const float *A;
  long lda;
  const float *B;
  long ldb;
  float *C;
  long ldc;
  float alpha, beta;
  const float *D;  // optional addend rows D[r >> dshift, :]
  long ldd;
  int dshift;
  int kchunk;      // K range per blockIdx.y (multiple of BK); == K when not split
  float *ws;       // split-K workspace (counters + partial tiles) or nullptr
  // cavs_embed_pull_sgemm (NN form only): row r of A is row int(pull_x[pull_rows[r]] * K) / K of the
  // table A points at (a negative id: a zero row); the workgroups of a row tile also leave the
  // rows they read in pull_copy (row stride ld_copy; each takes every tilesN-th k-tile) and those
  // of the first column tile the ids in pull_ids
  const int *pull_rows = nullptr;
  const float *pull_x = nullptr;
  float *pull_copy = nullptr;
  long ld_copy = 0;
  float *pull_ids = nullptr;
  // A block the caller knows about (cavs_gemm_desc::zero_kind and friends): the tiles it covers
  // run a shorter k range, or none
  int zkind = 0, zrows = 0, zcol = 0;
  // seg_rows > 0: the launch is several launches back to back, each padded to a multiple of 8 workgroups and dealt to the XCDs by
  // itself -- with one deal over all tiles the XCDs that hold those with less to do would finish early and the others set the time as
  // before: the row tiles inside the block up to column tile seg_cols, those up to seg_mixed (partly inside it), the other row
  // tiles, and what is left of the block (nothing but zeros to store)
  int seg_rows = 0, seg_cols = 0, seg_mixed = 0;
  const int *live = nullptr;  // cavs_gemm_desc::live
  int pad_block = 0, pad_used = 0;  // cavs_gemm_desc::pad_block, pad_used
  // an id per row of A as it is stored (of M, or of K where A is transposed): rows with equal ids, none below zero, are equal, and from
  // ids_from on they may well be
  const float *row_ids = nullptr;
  int ids_from = 0;
};

__device__ inline bool padding_column(const GemmArgs &g, int col) { return g.pad_block > 0 && col % g.pad_block >= g.pad_used; }

// The sizes a launch with `live` runs at: rows of C (TA = false) or K (TA = true), the known block's rows.
__device__ inline void apply_live(GemmArgs &g, bool TA, int splits) {
  if (!g.live) return;
  const int n = g.live[0];
  if (g.zkind) g.zrows = g.live[1];
  if (TA) {
    g.K = min(g.K, n);
    g.kchunk = max(32, ((g.K + splits - 1) / splits + 31) / 32 * 32);
  } else {
    g.M = min(g.M, n);
  }
}

// Remap the linear workgroup id so that ids that are consecutive after the remap
// were dispatched to the same XCD (hardware deals workgroups round-robin over 8 XCDs).
__device__ inline int xcd_remap(int l, int total) {
  constexpr int X = 8;
  int per = total / X, rem = total % X;
  int xcd = l % X, local = l / X;
  return xcd * per + (xcd < rem ? xcd : rem) + local;
}

// The part of K the tile at (m0, n0) of split `z` runs over.
template <int BM, int BN, bool TA, bool TB>
__device__ inline void tile_k_range(const GemmArgs &g, int m0, int n0, int z, int *beg, int *end) {
  int kbeg = z * g.kchunk;
  int kend = min(g.K, kbeg + g.kchunk);
  if (g.zkind == CAVS_GEMM_C_UNUSED) {  // rows below zrows of C are not wanted from column zcol on: left zero
    if (m0 + BM <= g.zrows && n0 >= g.zcol) kend = kbeg;
  } else if (g.zkind == CAVS_GEMM_A_ZERO) {  // rows below zrows of A (row-major M x K) are zero from k = zcol on
    if (!TA && m0 + BM <= g.zrows) kend = max(kbeg, min(kend, g.zcol));
  } else if (g.zkind == CAVS_GEMM_B_ZERO) {  // rows k < zrows of B (row-major K x N) are zero from column zcol on
    if (!TB && n0 >= g.zcol) kbeg = min(kend, max(kbeg, g.zrows / 32 * 32));
  }
  *beg = kbeg;
  *end = kend;
}

// Stores the TM x TN accumulators of a wavefront whose first row and column are m0 and n0.  THROUGH: partial sums past this
// XCD's L2, for workgroups anywhere in the same launch to read.
template <int TM, int TN, bool THROUGH = false>
__device__ inline void store_tile(const GemmArgs &g, const floatx16 (&acc)[TM][TN], int m0, int n0, int z, int lane) {
  const int khalf = lane >> 5;
  // C layout of the 32x32 accumulator: element r of lane l is row 8*(r/4) + 4*(l/32) + r%4,
  // column l%32.
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++) {
      const int col = n0 + 32 * j + (lane & 31);
      if (col >= g.N) continue;
      const int rbase = m0 + 32 * i + 4 * khalf;
      // the three forms of the store are chosen once per tile (the conditions are the same
      // for every lane), not once per element
      if (g.ws) {  // split K: park the partial sum, the reduce kernel finishes the job
        float *w = g.ws + (long)z * g.M * g.N + col;
        if constexpr (THROUGH) {
#pragma unroll
          for (int r = 0; r < 16; r++) {
            const int row = rbase + 8 * (r / 4) + (r % 4);
            if (row < g.M) __hip_atomic_store(w + (long)row * g.N, acc[i][j][r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          }
          continue;
        }
#pragma unroll
        for (int r = 0; r < 16; r++) {
          const int row = rbase + 8 * (r / 4) + (r % 4);
          if (row < g.M) w[(long)row * g.N] = acc[i][j][r];
        }
      } else if (g.beta == 0.f && !g.D) {
#pragma unroll
        for (int r = 0; r < 16; r++) {
          const int row = rbase + 8 * (r / 4) + (r % 4);
          if (row < g.M) g.C[row * g.ldc + col] = g.alpha * acc[i][j][r];
        }
      } else {
#pragma unroll
        for (int r = 0; r < 16; r++) {
          const int row = rbase + 8 * (r / 4) + (r % 4);
          if (row >= g.M) continue;
          float v = g.alpha * acc[i][j][r];
          if (g.beta != 0.f) v += g.beta * g.C[row * g.ldc + col];
          if (g.D) v += g.D[(long)(row >> g.dshift) * g.ldd + col];
          g.C[row * g.ldc + col] = v;
        }
      }
    }
}

}  // namespace cavs
