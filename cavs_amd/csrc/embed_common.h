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
__device__ inline void embed_bwd_block(float *__restrict__ dtable, const float *__restrict__ ids, const float *__restrict__ dy,
                                       long ld_dy, int parts, long part_stride, float *__restrict__ copy, long ld_copy, int n, int E,
                                       int bx, int by) {
  __shared__ float part[4][kEmbedCols];
  const int row0 = bx * kEmbedRows, tid = threadIdx.x;
  const int rows = min(kEmbedRows, n - row0);
  const int q = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, c = by * kEmbedCols + lane;
  constexpr int U = kEmbedRows / 4;  // rows per wavefront, all in flight
  const int r0 = q * U;
  const int mine = lane < rows ? (int)(ids[row0 + lane] * (float)E) : -1 - lane;  // this lane's row of the table, as its first float
  float v[U];
  if (c < E) {
#pragma unroll
    for (int u = 0; u < U; u++) v[u] = r0 + u < rows ? dy[(long)(row0 + r0 + u) * ld_dy + c] : 0.f;
  }
  // occurrences of this lane's id, counted at its first occurrence only; the most frequent one, ties: the earliest row
  int count = 0;
  bool first = lane < rows;
#pragma unroll
  for (int r = 0; r < kEmbedRows; r++) {
    const bool same = __builtin_amdgcn_readlane(mine, r) == mine;
    count += same;
    if (same && r < lane) first = false;
  }
  int key = first ? count * 64 + (63 - lane) : 0;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) key = max(key, __shfl_xor(key, o, 64));
  key = __builtin_amdgcn_readfirstlane(key);
  const bool combine = key / 64 > 1;
  const int hot = __builtin_amdgcn_readlane(mine, 63 - (key & 63));
  float sum = 0.f;
  if (c < E) {
    if (parts == 2) {  // the usual split: both parts' loads in flight together
      float w[U];
      const float *dz = dy + part_stride;
#pragma unroll
      for (int u = 0; u < U; u++) w[u] = r0 + u < rows ? dz[(long)(row0 + r0 + u) * ld_dy + c] : 0.f;
#pragma unroll
      for (int u = 0; u < U; u++) v[u] += w[u];
    } else {
      for (int z = 1; z < parts; z++) {
        const float *dz = dy + z * part_stride;
        float w[U];
#pragma unroll
        for (int u = 0; u < U; u++) w[u] = r0 + u < rows ? dz[(long)(row0 + r0 + u) * ld_dy + c] : 0.f;
#pragma unroll
        for (int u = 0; u < U; u++) v[u] += w[u];
      }
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
      if (combine && o == hot) sum += v[u];  // in row order
      else unsafeAtomicAdd(dtable + o + c, v[u]);
    }
  }
  if (!combine) return;  // the same for the whole workgroup
  part[q][lane] = sum;
  __syncthreads();
  if (q == 0 && c < E) unsafeAtomicAdd(dtable + hot + c, ((part[0][lane] + part[1][lane]) + part[2][lane]) + part[3][lane]);
}

}  // namespace cavs
#endif
