// The chunk sums of a matrix' columns, shared by cavs_colsum_blocks and by the grouped products' launch that
// takes them along (cavs_sgemm_group_once).
#ifndef CAVS_CSRC_COLSUM_COMMON_H_
#define CAVS_CSRC_COLSUM_COMMON_H_

#include "common.h"

namespace cavs {

struct ColsumParts {
  float *part;        // [chunks][w]
  const float *inp;   // [n][ld]
  long ld;
  int n, w, rows, chunks;  // rows of a chunk
};
inline int colsum_chunks(int n) {
  const int c = (n + 127) / 128;
  return c < 1 ? 1 : (c > 32 ? 32 : c);
}
inline ColsumParts colsum_job(float *part, const float *inp, long ld, int n, int w) {
  const int chunks = colsum_chunks(n);
  return {part, inp, ld, n, w, ((n + chunks - 1) / chunks + 3) / 4 * 4, chunks};
}

// columns 64 bx .. of chunk `chunk` by four wavefronts
__device__ inline void colsum_part_block(const ColsumParts &j, int bx, int chunk, float (*s)[64]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = bx * 64 + lane;
  const int r0 = chunk * j.rows, r1 = min(j.n, r0 + j.rows);
  float a0 = 0.f, a1 = 0.f;
  if (col < j.w) {
    int r = r0 + wave;
    for (; r + 4 < r1; r += 8) {
      a0 += j.inp[(long)r * j.ld + col];
      a1 += j.inp[(long)(r + 4) * j.ld + col];
    }
    for (; r < r1; r += 4) a0 += j.inp[(long)r * j.ld + col];
  }
  s[wave][lane] = a0 + a1;
  __syncthreads();
  if (wave == 0 && col < j.w) j.part[(long)chunk * j.w + col] = (s[0][lane] + s[1][lane]) + (s[2][lane] + s[3][lane]);
}

}  // namespace cavs
#endif
