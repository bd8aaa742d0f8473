// The embedding gradient's scatter-add, shared by cavs_embed_bwd and by the grouped products'
// launch that reduces K-split partials (which feeds it the product's partials directly).
#ifndef CAVS_CSRC_EMBED_COMMON_H_
#define CAVS_CSRC_EMBED_COMMON_H_

#include "common.h"

namespace cavs {

// Scatter-add of dy rows into the table.  A workgroup takes 64 consecutive rows and 64 columns
// (row chunk bx, column chunk by).
// Parse trees look up one and the same table row for every internal vertex, and atomic adds to
// one address serialise, so the workgroup first finds the id that occurs most often among its
// rows (its "hot" id), adds those rows up (each wavefront its 16 rows in registers, then the
// four partial sums in wavefront order) and issues one atomic add per column for them; every
// other row goes to the table with an atomic add of its own.  Each wavefront finds the hot id by itself, a
// row to a lane, the other rows' ids broadcast one after the other: 64 compares and a reduction by
// shuffles (through LDS, with one thread picking the maximum, 907 rows of 300 columns took 11.7 us, 8.9 now,
// launch included).
// dy is the sum of `parts` arrays `part_stride` floats apart, added in index order (one array:
// the plain case); when `copy` is given the summed value is also stored there (row stride ld_copy).
constexpr int kEmbedRows = 64, kEmbedCols = 64;
// Rows of a wavefront from p on, one column to a lane, as workgroups of the same launch have left them, on any XCD (past this
// one's caches).  The row's address is a scalar: no register of a lane holds one.
struct ThroughRows {
  int ld, last, col;  // floats between rows, last row there is, the lane's byte
  template <int U>
  __device__ inline void load(const float *p, float (&v)[U]) const {
    constexpr int SC1 = 16;
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p), 0, 0xffffffffu, 0x00020000);
#pragma unroll
    for (int u = 0; u < U; u++) v[u] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, col, min(u, last) * ld * 4, SC1));
  }
};

// this lane's row of the table, as its first float (none: below zero, and nobody else's)
__device__ inline int embed_row(const float *__restrict__ ids, int n, int E, int bx) {
  const int lane = threadIdx.x & 63, row0 = bx * kEmbedRows;
  return lane < n - row0 ? (int)(ids[row0 + lane] * (float)E) : -1 - lane;
}
struct EmbedHot {
  int row;       // the most frequent row among the workgroup's lookups, ties: the earliest
  bool combine;  // it occurs more than once (the same for the whole workgroup)
};
__device__ inline EmbedHot embed_hot(int mine) {
  const int lane = threadIdx.x & 63;
  // occurrences of this lane's id, counted at its first occurrence only
  int count = 0;
  bool first = mine >= 0;
#pragma unroll 16
  for (int r = 0; r < kEmbedRows; r++) {
    const bool same = __builtin_amdgcn_readlane(mine, r) == mine;
    count += same;
    if (same && r < lane) first = false;
  }
  int key = first ? count * 64 + (63 - lane) : 0;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) key = max(key, __shfl_xor(key, o, 64));
  key = __builtin_amdgcn_readfirstlane(key);
  return {__builtin_amdgcn_readlane(mine, 63 - (key & 63)), key / 64 > 1};
}
// `hot`: called once dy's first part has been asked for
template <bool THROUGH, class Hot>
__device__ inline void embed_bwd_rows(float *__restrict__ dtable, int mine, Hot hot_of, const float *__restrict__ dy, long ld_dy, int parts,
                                      long part_stride, float *__restrict__ copy, long ld_copy, int n, int E, int bx, int by) {
  __shared__ float part[4][kEmbedCols];
  const int row0 = bx * kEmbedRows, tid = threadIdx.x;
  const int rows = min(kEmbedRows, n - row0);
  const int q = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, c = by * kEmbedCols + lane;
  constexpr int U = kEmbedRows / 4;  // rows per wavefront, all in flight
  const int r0 = q * U;
  float v[U];
  const float *p = dy + (long)(row0 + r0) * ld_dy;
  const bool on = c < E && r0 < rows;
  const ThroughRows through{(int)ld_dy, rows - 1 - r0, 4 * c};
  if (on) {
    if constexpr (THROUGH) {
      through.load(p, v);
    } else {
#pragma unroll
      for (int u = 0; u < U; u++) v[u] = r0 + u < rows ? p[(long)u * ld_dy + c] : 0.f;
    }
  }
  const EmbedHot hot = hot_of();
  float sum = 0.f;
  if (on) {
    constexpr int D = THROUGH ? 3 : 1;  // parts in flight, besides the first
    for (int z = 1; z < parts; z += D) {
      p += part_stride;
      float w[D][U];
#pragma unroll
      for (int k = 0; k < D; k++) {
        if constexpr (THROUGH) {
          through.load(p + (z + k < parts ? k : 0) * part_stride, w[k]);
        } else {
#pragma unroll
          for (int u = 0; u < U; u++) w[k][u] = r0 + u < rows ? p[(long)u * ld_dy + c] : 0.f;
        }
      }
#pragma unroll
      for (int k = 0; k < D; k++) {
        if (z + k >= parts) break;
#pragma unroll
        for (int u = 0; u < U; u++) v[u] += w[k][u];
      }
      p += (D - 1) * part_stride;
    }
    if (copy) {
#pragma unroll
      for (int u = 0; u < U; u++)
        if (r0 + u < rows) copy[(long)(row0 + r0 + u) * ld_copy + c] = v[u];
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (r0 + u >= rows) continue;
      const int o = __builtin_amdgcn_readlane(mine, r0 + u);
      if (hot.combine && o == hot.row) sum += v[u];  // in row order
      else unsafeAtomicAdd(dtable + o + c, v[u]);
    }
  }
  if (!hot.combine) return;
  part[q][lane] = sum;
  __syncthreads();
  if (q == 0 && c < E) unsafeAtomicAdd(dtable + hot.row + c, ((part[0][lane] + part[1][lane]) + part[2][lane]) + part[3][lane]);
}
__device__ inline void embed_bwd_block(float *__restrict__ dtable, const float *__restrict__ ids, const float *__restrict__ dy,
                                       long ld_dy, int parts, long part_stride, float *__restrict__ copy, long ld_copy, int n, int E,
                                       int bx, int by) {
  const int mine = embed_row(ids, n, E, bx);
  embed_bwd_rows<false>(dtable, mine, [&] { return embed_hot(mine); }, dy, ld_dy, parts, part_stride, copy, ld_copy, n, E, bx, by);
}

}  // namespace cavs
#endif
