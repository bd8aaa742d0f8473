// fp32 products on the bf16 matrix pipe, in full fp32 precision.
//
// The fp32 MFMA does 256 multiply-adds x 2 per clock and CU, the bf16 one sixteen times that.  A
// float is exactly the sum of three bf16 numbers: h = bf16(x), m = bf16(x - h), l = x - h - m (both
// differences are exact, eight significant bits each), so a product is the sum of nine bf16 products,
// each of them exact in the fp32 accumulator.  (Splitting a number into a sum of shorter ones whose
// products are exact: Dekker, "A floating-point technique for extending the available precision", 1971;
// into bf16 parts for matrix units: Henry, Tang and Heinecke, "Leveraging the bfloat16 artificial intelligence
// datatype for higher-precision computations", 2019.)  The six of weight 2^-16 and above are added up; the
// other three are below 2^-26 of the product, a quarter of the rounding that one fp32 addition
// makes.  Six bf16 MFMAs take 6/16 of the matrix pipe's time for the fp32 product, and because an
// instruction adds 16 values of k before it rounds, the sum rounds less often than the fp32 chain.
//
// What the pipe drops: it rounds a sum to nearest, but an addend of less than about an eighth of the
// accumulator's last place is lost in it (1 + 16 x 2^-27 is 1), and the parts m and l of a long sum's
// terms are such addends.  Where they all push one way -- constants, values on a grid -- a chain of 2048
// of K was up to seven times further off than the fp32 pipe.  So a chain of additions ends after kSplitChain = 256
// of K and goes into a second set of accumulators by ordinary additions; a product of up to 512 of K on
// the large tile is one chain, which is no further off than the fp32 pipe there.  The second set costs the
// large tile its third workgroup per CU (232 registers instead of 167) and 1 to 5 % of its rate; storing
// and reloading C between chains instead cost 20 %.
//
// An infinite operand (infinity - infinity while splitting) or a finite one whose h rounds to infinity makes
// NaN; so do NaN operands.  A wavefront whose results are not all finite computes them again on the fp32 MFMA
// (unsplit_tile): 8192^3 with a NaN in every row takes 26 ms, with one 17, without 6.  Parts below 2^-133
// are no bf16 numbers: of an operand below 2^-110 bits of that weight are lost.
//
// A workgroup of 4 wavefronts (2 x 2) computes a BM x BN tile, BK of k at a time (two LDS buffers, one
// barrier per step).  Operands are split on their way into LDS: row x of an operand tile is 2 BK bytes
// per part, its 16-byte pieces permuted by x so that sixteen lanes reading the same k of sixteen rows
// touch all 64 banks once (without it: a third of the LDS time).  While a step multiplies, the values of
// the next one are converted and those of the one behind it are under way; the conversions (4.5
// vector instructions a value) run in the shadow of the MFMAs of the two or three workgroups a CU holds.
// What bounds it is power: with random operands the clock falls to 1.63 - 1.77 GHz (NN and NT below; 2.0 for TN), with
// operands of zeros the same instructions run at 2.39 GHz and 262 - 290 TFLOP/s.  bf16 MFMAs alone, from registers, sustain
// 1.63 - 1.88 PFLOP/s here (1.75 GHz), i.e. 270 - 310 TFLOP/s of these products.
//
// us (TFLOP/s)                  fp32 MFMA, 128 x 128 x 16      this
//   NN  8192 x  8192 x  8192    8198 (134)                     5766 (191)
//   NT 73000 x  1024 x  4096    4763 (129)                     3056 (200)
//   TN  1024 x  4096 x 73000    4664 (131)                     3402 (180)
//   NN  7088 x 10000 x   512     688 (105)                      407 (178)
//   NN  2368 x  2048 x   300    34.2 (85)    (64 x 64 tiles)   27.1 (107)
//   TN   304 x  2048 x  2368    43.2 (68)                      34.7 (85)
// Operands that are not k-contiguous cost instructions (a load per value, 230 a step and wavefront with their
// addresses): read through buffer descriptors, on one card, us before / now: NN 8192 5920 / 5681, NN 73000 x 4096 x 1024
// 3365 / 3226, NN 7088 409 / 391, TN 73000 3470 / 3335; NT, which has none, 3132 / 3125.  Tried: parts read a
// step ahead from three buffers (NN + 2 %, NT + 2 %, TN - 4 %: a third of the cycles less, a clock as much lower).
// 2-norm of the error against 64 bits over that of the product, fp32 MFMA / this, 1e-7: operands from U(-1, 1),
// from U(0, 1), and all of the form (eight bits) (1 + 2^-10 + 2^-11):
//   NN  8192    16.2 / 2.7   11.9 / 0.8   11.8 / 1.4        NT 73000    11.5 / 2.5   8.5 / 0.7    8.4 / 1.3
//   TN  1024    27.9 / 3.8   13.7 / 1.3   16.6 / 1.7        NN  7088     4.1 / 3.4   3.1 / 2.4    3.0 / 3.3
//   NN  2368     3.1 / 2.2    2.6 / 1.6    2.7 / 1.6        TN   304     3.9 / 2.4   1.4 / 0.7    1.4 / 1.2
#pragma once
#include <type_traits>

#include "gemm_common.h"

namespace cavs {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx8 __attribute__((ext_vector_type(8)));

// bf16 of two floats (round to nearest), the first in the low half
__device__ inline unsigned bf16_pair(float x, float y) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(unsigned, __builtin_convertvector((f2{x, y}), b2));
}

__device__ inline void split_pair(float x, float y, unsigned *h, unsigned *m, unsigned *l) {
  *h = bf16_pair(x, y);
  x -= __uint_as_float(*h << 16);
  y -= __uint_as_float(*h & 0xffff0000u);
  *m = bf16_pair(x, y);
  x -= __uint_as_float(*m << 16);
  y -= __uint_as_float(*m & 0xffff0000u);
  *l = bf16_pair(x, y);
}

// where the 16-byte piece of row x that holds k = 8 oct .. 8 oct + 7 lies in a part of a tile BK deep.  Rows of 32 bytes: reads
// take 4.2 cycles a wavefront and instruction with either rule (8.0 unpermuted); eight values of k written by
// 64 rows at once take 13 with the second and 16 with the first.
template <int BK, bool KC>
__device__ inline int split_at(int x, int oct) {
  if (BK == 16) return x * 32 + ((oct ^ ((x >> 3) & 1) ^ (KC ? 0 : (x >> 2) & 1)) << 4);
  return x * 64 + ((oct ^ ((x >> 2) & 3)) << 4);
}

// Loader of one BX x BK operand tile: units of one x and U values of k, NU per thread.  KC: k is the
// contiguous index in memory and a unit is 16 bytes of it; otherwise a unit is eight rows of one
// column.  An x outside the operand reads the last one instead (what it leads to is not stored);
// only k is checked, and only where the step is not wholly inside the k range.
// PULL (k-contiguous): rows are looked up (GemmArgs::pull_*); a row without an id reads the table's first, and is zero.
template <int BX, int BK, bool KC, bool VEC, bool DESC, bool PULL = false>
struct SplitLoader {
  static constexpr int U = KC || BX * BK < 8 * kThreads ? 4 : 8, NU = BX * BK / U / kThreads, PER = BK / U;
  using Off = std::conditional_t<BX == 64, size_t, unsigned>;  // (the large tile's registers are full: its rows are below 32 MB)
  Off boff[NU];  // bytes from the tile's first element (k-contiguous: at k = U unit)
  int unit[NU];
  int at[NU];  // byte of a part the unit goes to

  __device__ inline void prepare(long ld, int x0, int X, int tid) {
#pragma unroll
    for (int i = 0; i < NU; i++) {
      if constexpr (KC) {
        const int u = tid + kThreads * i;
        unit[i] = u % PER;
        boff[i] = (Off)min(u / PER, X - 1 - x0) * (Off)(ld * 4) + 16u * unit[i];
        at[i] = split_at<BK, KC>(u / PER, unit[i] >> 1) + 8 * (unit[i] & 1);
      } else {
        unit[i] = __builtin_amdgcn_readfirstlane(tid / BX + (kThreads / BX) * i);  // (BX is a multiple of 64)
        boff[i] = 4u * (unsigned)min(tid % BX, X - 1 - x0);
        at[i] = split_at<BK, KC>(tid % BX, unit[i] * U / 8) + (U == 4 ? 8 * (unit[i] & 1) : 0);
      }
    }
  }

  // Row x0 + r of the operand is the table row that starts at float int(id * K) (EmbeddingLookup's
  // offset), id = px[rows[x0 + r]]; a negative id is a zero row.
  bool in[PULL ? NU : 1];  // the row has an id
  bool all_in = true;      // every row of this wavefront has
  long one = -1;  // the row this wavefront's units are all of, if they are; -2: it has none
  __device__ inline void prepare_pull(const GemmArgs &g, int x0, int tid, float *ids_out) {
    static_assert(!PULL || KC, "looked-up rows are k-contiguous");
#pragma unroll
    for (int i = 0; i < NU; i++) {
      const int u = tid + kThreads * i, x = u / PER, gx = x0 + x;
      unit[i] = u % PER;
      at[i] = split_at<BK, KC>(x, unit[i] >> 1) + 8 * (unit[i] & 1);
      long off = -1;
      if (gx < g.M) {
        const float id = g.pull_x[g.pull_rows[gx]];
        off = max((long)(int)(id * (float)g.K), -1L);  // (any row without an id: -1, so that -2 says something else)
        if (ids_out && unit[i] == 0) ids_out[gx] = id;
      }
      if (i == 0) one = __builtin_amdgcn_readfirstlane(gx < g.M ? (int)off : -2);  // (rows ascend: beyond the last, all of them are)
      if (!__all(off == one || gx >= g.M)) one = -1;
      in[i] = off >= 0 || gx >= g.M;
      all_in &= __all(in[i]);
      boff[i] = 4 * ((Off)(off >= 0 ? off : 0) + U * unit[i]);
    }
  }

  // P: the tile's first element at k = 0; k0 and kend are wave-uniform.  DESC: a whole step is read through a buffer descriptor, the
  // step's address in scalar registers and a row's offset in a vector register that never changes: no vector
  // instructions for addresses.
  template <bool WHOLE>
  __device__ inline void load(float (&v)[NU][U], const float *__restrict__ P, long ld, int k0, int kend) const {
    if constexpr (WHOLE && DESC && !PULL && (!KC || VEC)) {
      const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(P + (KC ? (long)k0 : (long)k0 * ld)), 0, 0xffffffffu, 0x00020000);
#pragma unroll
      for (int i = 0; i < NU; i++) {
        if constexpr (KC) {
          typedef float f4 __attribute__((ext_vector_type(4)));
          const f4 a = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)boff[i], 0, 0));
#pragma unroll
          for (int j = 0; j < 4; j++) v[i][j] = a[j];
        } else {
#pragma unroll
          for (int j = 0; j < U; j++)
            v[i][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)boff[i], (int)((U * unit[i] + j) * (unsigned)(ld * 4)), 0));
        }
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < NU; i++) {
      if constexpr (KC) {
        const float *q = reinterpret_cast<const float *>(reinterpret_cast<const char *>(P + k0) + boff[i]);
        if constexpr (WHOLE && VEC) {
          const float4 a = *reinterpret_cast<const float4 *>(q);
          v[i][0] = a.x, v[i][1] = a.y, v[i][2] = a.z, v[i][3] = a.w;
        } else {
          const int left = kend - k0 - U * unit[i];
#pragma unroll
          for (int j = 0; j < U; j++) v[i][j] = (WHOLE || j < left) ? q[j] : 0.f;
        }
      } else {
        const int k = k0 + U * unit[i];
        const char *q = reinterpret_cast<const char *>(P + (long)k * ld);
#pragma unroll
        for (int j = 0; j < U; j++) {
          v[i][j] = (WHOLE || k + j < kend) ? *reinterpret_cast<const float *>(q + boff[i]) : 0.f;
          q += ld * 4;
        }
      }
    }
  }

  __device__ inline void store(float (&v)[NU][U], char *__restrict__ S) const {
    if constexpr (PULL) {
      if (!all_in) {
#pragma unroll
        for (int i = 0; i < NU; i++)
#pragma unroll
          for (int j = 0; j < U; j++) v[i][j] = in[i] ? v[i][j] : 0.f;
      }
    }
#pragma unroll
    for (int i = 0; i < NU; i++) {
      unsigned h[U / 2], m[U / 2], l[U / 2];
#pragma unroll
      for (int j = 0; j < U / 2; j++) split_pair(v[i][2 * j], v[i][2 * j + 1], h + j, m + j, l + j);
      if constexpr (U == 4) {
        *reinterpret_cast<uint2 *>(S + at[i]) = make_uint2(h[0], h[1]);
        *reinterpret_cast<uint2 *>(S + at[i] + BX * BK * 2) = make_uint2(m[0], m[1]);
        *reinterpret_cast<uint2 *>(S + at[i] + 2 * BX * BK * 2) = make_uint2(l[0], l[1]);
      } else {
        *reinterpret_cast<uint4 *>(S + at[i]) = make_uint4(h[0], h[1], h[2], h[3]);
        *reinterpret_cast<uint4 *>(S + at[i] + BX * BK * 2) = make_uint4(m[0], m[1], m[2], m[3]);
        *reinterpret_cast<uint4 *>(S + at[i] + 2 * BX * BK * 2) = make_uint4(l[0], l[1], l[2], l[3]);
      }
    }
  }
};

// K of one chain of additions on the bf16 pipe (see above)
constexpr int kSplitChain = 256;

// What the fp32 pipe makes of a wavefront's TM x TN tiles over [kbeg, kend): the operands as they are, straight
// from memory.  Only for results that came out infinite or NaN (split_tile).
template <int TM, int TN, bool TA, bool TB, bool PULL>
__device__ inline void unsplit_tile(const GemmArgs &g, int row, int col, int kbeg, int kend, int lane, floatx16 (&acc)[TM][TN]) {
  const int x = lane & 31, half = lane >> 5;
  const float *pa[TM], *pb[TN];
  bool on[TM];
#pragma unroll
  for (int i = 0; i < TM; i++) {
    const int m = min(row + 32 * i + x, g.M - 1);
    on[i] = true;
    if constexpr (PULL) {
      const long off = (long)(int)(g.pull_x[g.pull_rows[m]] * (float)g.K);
      on[i] = off >= 0;
      pa[i] = g.A + (on[i] ? off : 0);
    } else {
      pa[i] = TA ? g.A + m : g.A + (long)m * g.lda;
    }
  }
#pragma unroll
  for (int j = 0; j < TN; j++) {
    const int n = min(col + 32 * j + x, g.N - 1);
    pb[j] = TB ? g.B + (long)n * g.ldb : g.B + n;
  }
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
  constexpr int U = 8;  // pairs of k in flight
  for (int k0 = kbeg; k0 < kend; k0 += 2 * U) {
    float a[U][TM], b[U][TN];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int k = k0 + 2 * u + half, kc = min(k, kend - 1);
#pragma unroll
      for (int i = 0; i < TM; i++) a[u][i] = pa[i][TA ? (long)kc * g.lda : kc];
#pragma unroll
      for (int j = 0; j < TN; j++) b[u][j] = pb[j][TB ? kc : (long)kc * g.ldb];
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const bool in = k0 + 2 * u + half < kend;
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(in && on[i] ? a[u][i] : 0.f, in ? b[u][j] : 0.f, acc[i][j], 0, 0, 0);
    }
  }
#pragma unroll
  for (int j = 0; j < TN; j++)
    if (padding_column(g, col + 32 * j + x))
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
}

// ------------------------------------------------------------------ rows that are all the same
// The inner vertices of a parse tree carry no word: they all look one table row up, and in a batch's rows they stand together, behind
// the leaves.  So the lower half of x * W's row tiles hold one and the same row, the d W of those vertices is one row times the
// sum of their gradients, and what they send to the table is that sum times W^T.  A tile finds out by itself (row_ids: rows
// with equal ids are equal) and does a vector's work in fp32 where it would do a matrix's:
//   x * W      one row times its columns of B, written to every row                    (same_rows_product)
//   A^T * B    the sum of B's rows over its part of K, then one step of K = 1 as MFMA  (in split_tile)
//   A * B^T    for the table: the sum of A's rows times its columns of B               (summed_rows_product)
// Sums that leave a float's range are not used: A^T * B makes NaN of them, which unsplit_tile computes again row by row, A * B^T takes
// the general way.
// What bounds such a tile are trips to memory, so its loads are all in flight at once.  64 trees, H = 512 (1217 leaves, 1153 inner
// vertices), us a launch: x * W 30.4 -> 20.5, the deferred products 75 -> 64; 256 trees x * W 73.5 -> 47; Tree-LSTM steps of 64
// trees 10250 -> 9550 (32 of them, with the resident rounds' change before).
// The sums are shorter than the chains they replace, and in pairs.  2-norm of the error against 64 bits over that of the result, 2370 rows of
// 300, 2048 columns, normal operands / operands from U(0, 1), before and now, 1e-7: x W 2.3 -> 1.9 / 1.7 -> 1.4, d W 2.4 -> 2.0 / 0.9 -> 0.6,
// the table's gradient 10.3 -> 2.2 / 0.72 -> 0.67.

// Whether ids[first .. end) are one and the same (the whole workgroup asks; every wavefront finds the same)
__device__ inline bool same_ids(const float *__restrict__ ids, int first, int end) {
  const float id = ids[first];
  bool same = id >= 0.f;
  for (int i = first + (threadIdx.x & 63); i < end; i += 64) same &= ids[i] == id;
  return __all(same);
}

// One element of the product's result, or of its part of it
template <bool THROUGH>
__device__ inline void put_result(const GemmArgs &g, int z, int row, int col, float v) {
  if (!g.ws) {
    g.C[row * g.ldc + col] = g.alpha * v;
    return;
  }
  float *w = g.ws + ((long)z * g.M + row) * g.N + col;
  if constexpr (THROUGH) __hip_atomic_store(w, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else *w = v;
}

constexpr int kSameK = 4096;  // the row has room in the tile's LDS

// C's rows m0 .. m0 + BM, columns n0 .. n0 + BN: `row` (K floats) times B, in every row.  beta = 0, K not split.  A thread has C of the
// columns and every PARTS-th of K, as many loads in flight as there are registers for: one trip to memory behind the other is all
// the time this takes.
template <int BM, int BN, bool VEC>
__device__ __forceinline__ void same_rows_product(const GemmArgs &g, const float *__restrict__ row, int m0, int n0, char *__restrict__ S) {
  constexpr int C = VEC ? 4 : 1, ACROSS = BN / C, PARTS = kThreads / ACROSS, U = VEC ? 12 : 32;
  float *a = reinterpret_cast<float *>(S), *part = a + kSameK;  // [kSameK], [PARTS][BN]
  const int tid = threadIdx.x, c = C * (tid % ACROSS), q = tid / ACROSS;
  const float *b = g.B + min(n0 + c, g.N - C);
  float acc[C] = {}, v[U][C];
  auto load = [&](int k0) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      const float *at = b + (long)min(k0 + q + u * PARTS, g.K - 1) * g.ldb;
      if constexpr (VEC) {
        const float4 t = *reinterpret_cast<const float4 *>(at);
        v[u][0] = t.x, v[u][1] = t.y, v[u][2] = t.z, v[u][3] = t.w;
      } else {
        v[u][0] = *at;
      }
    }
  };
  load(0);
  for (int k = tid; k < g.K; k += kThreads) a[k] = row[k];
  __syncthreads();
  for (int k0 = 0; k0 < g.K; k0 += U * PARTS) {
    if (k0 > 0) load(k0);
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int k = k0 + q + u * PARTS;
      const float x = k < g.K ? a[k] : 0.f;
#pragma unroll
      for (int j = 0; j < C; j++) acc[j] = k < g.K ? fmaf(x, v[u][j], acc[j]) : acc[j];
    }
  }
#pragma unroll
  for (int j = 0; j < C; j++) part[q * BN + c + j] = acc[j];
  __syncthreads();
  // the parts' sums, a column to a thread, in their order; then every row
  if (tid < BN) {
    float t = 0.f;
    for (int p = 0; p < PARTS; p++) t += part[p * BN + tid];
    a[tid] = padding_column(g, n0 + tid) ? 0.f : g.alpha * t;
  }
  __syncthreads();
  for (int r = q; r < BM && m0 + r < g.M; r += PARTS) {
    float *to = g.C + (long)(m0 + r) * g.ldc + n0 + c;
    if (VEC && g.ldc % 4 == 0 && n0 + c < g.N && (reinterpret_cast<uintptr_t>(to) & 15) == 0) {
      *reinterpret_cast<float4 *>(to) = *reinterpret_cast<const float4 *>(a + c);
    } else {
#pragma unroll
      for (int j = 0; j < C; j++)
        if (n0 + c + j < g.N) to[j] = a[c + j];
    }
  }
}

// The rows of a tile that were looked up, on into pull_copy: the column tiles that run share them, every tilesN-th step of K each.  (Behind
// the product, when the rows are near: among its loads the stores' conditions had every wait be for everything.)
template <int BM, int BN, int BK, bool VEC>
__device__ __forceinline__ void copy_looked_up(const GemmArgs &g, int m0, int n0) {
  const int tilesN = (g.N + BN - 1) / BN;
  const int active = (g.zkind == CAVS_GEMM_C_UNUSED && m0 + BM <= g.zrows) ? min(tilesN, (g.zcol + BN - 1) / BN) : tilesN;
  constexpr int U = VEC ? 4 : 1;
  const int x = threadIdx.x / (BK / U), k_ = threadIdx.x % (BK / U) * U;
  for (int k0 = n0 / BN * BK; k0 < g.K; k0 += BK * active)
    for (int r = x; r < BM; r += kThreads / (BK / U)) {
      const int row = m0 + r, k = k0 + k_;
      if (row >= g.M || k >= g.K) continue;
      const long off = (long)(int)(g.pull_x[g.pull_rows[row]] * (float)g.K);
      float *to = g.pull_copy + (long)row * g.ld_copy + k;
      if constexpr (VEC) *reinterpret_cast<float4 *>(to) = off >= 0 ? *reinterpret_cast<const float4 *>(g.A + off + k) : make_float4(0.f, 0.f, 0.f, 0.f);
      else *to = off >= 0 ? g.A[off + k] : 0.f;
    }
}

// sixteen values added up in pairs
__device__ inline float4 pairs(float4 (&v)[16]) {
#pragma unroll
  for (int n = 8; n > 0; n /= 2)
#pragma unroll
    for (int i = 0; i < n; i++) v[i].x += v[i + n].x, v[i].y += v[i + n].y, v[i].z += v[i + n].z, v[i].w += v[i + n].w;
  return v[0];
}

// Sixteen rows from p on, a float4 of each to a lane at byte `at` of a row: the rows' offsets are scalars
__device__ inline void sixteen_rows(const float *p, int ld, int last, int at, float4 (&v)[16]) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p), 0, 0xffffffffu, 0x00020000);
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const f4 a = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(r, at, max(min(i, last), 0) * ld * 4, 0));
    v[i] = make_float4(a[0], a[1], a[2], a[3]);
  }
}

// Rows m0 .. m0 + 64 of A (M x K) summed, times rows n0 .. n0 + 64 of B (N x K), over [kbeg, kend): the first row of the tile of C, and
// zeros in the others.  kbeg, kend, lda, ldb are multiples of 4, A and B 16-byte aligned.  False, with nothing stored, where a result is not
// finite: the sum of the rows may pass a float's range where every row's product is inside it.
template <bool THROUGH>
__device__ __forceinline__ bool summed_rows_product(const GemmArgs &g, int m0, int n0, int z, int kbeg, int kend, char *__restrict__ S) {
  constexpr int KB = 1024, ROWS = 16;  // k at a time; rows of A and of B to a wavefront
  float *s = reinterpret_cast<float *>(S);  // [4][KB], the sums in the first
  float *out = s + 4 * KB;                  // [64]
  const int tid = threadIdx.x, lane = tid & 63, q = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ra = min(m0 + ROWS * q, g.M - 1), rb = min(n0 + ROWS * q, g.N - 1);  // (a wavefront beyond the last row adds nothing, or is not stored)
  const int rows = g.M - (m0 + ROWS * q), cols = g.N - 1 - rb;
  const float *A = g.A + (long)ra * g.lda, *B = g.B + (long)rb * g.ldb;
  const int lda = (int)g.lda, ldb = (int)g.ldb;
  float acc[ROWS];
#pragma unroll
  for (int e = 0; e < ROWS; e++) acc[e] = 0.f;
  for (int k0 = kbeg; k0 < kend; k0 += KB) {
    const int len = min(KB, kend - k0);
    __syncthreads();
    for (int k = 4 * lane; k < len; k += 256) {
      float4 v[ROWS];
      sixteen_rows(A + k0, lda, rows - 1, 4 * k, v);
#pragma unroll
      for (int r = 0; r < ROWS; r++)
        if (r >= rows) v[r] = make_float4(0.f, 0.f, 0.f, 0.f);
      *reinterpret_cast<float4 *>(s + q * KB + k) = pairs(v);
    }
    __syncthreads();
    for (int k = 4 * tid; k < len; k += 4 * kThreads) {
      float4 t = *reinterpret_cast<const float4 *>(s + k);
#pragma unroll
      for (int p = 1; p < 4; p++) {
        const float4 o = *reinterpret_cast<const float4 *>(s + p * KB + k);
        t.x += o.x, t.y += o.y, t.z += o.z, t.w += o.w;
      }
      *reinterpret_cast<float4 *>(s + k) = t;
    }
    __syncthreads();
    for (int k = 4 * lane; k < len; k += 256) {
      const float4 t = *reinterpret_cast<const float4 *>(s + k);
      float4 v[ROWS];
      sixteen_rows(B + k0, ldb, cols, 4 * k, v);
#pragma unroll
      for (int e = 0; e < ROWS; e++) acc[e] = fmaf(t.w, v[e].w, fmaf(t.z, v[e].z, fmaf(t.y, v[e].y, fmaf(t.x, v[e].x, acc[e]))));
    }
  }
  // the lanes' sums of sixteen columns: halves are exchanged until a lane holds one
#pragma unroll
  for (int n = ROWS / 2; n > 0; n /= 2)
#pragma unroll
    for (int e = 0; e < n; e++) {
      const bool up = lane & (4 * n);
      const float give = up ? acc[e] : acc[e + n], keep = up ? acc[e + n] : acc[e];
      acc[e] = keep + __shfl_xor(give, 4 * n, 64);
    }
  acc[0] += __shfl_xor(acc[0], 2, 64);
  acc[0] += __shfl_xor(acc[0], 1, 64);
  if ((lane & 3) == 0) out[ROWS * q + (lane >> 2)] = acc[0];
  __syncthreads();
  const float sum = out[lane];  // (every wavefront looks at all of them)
  if (!__all(n0 + lane >= g.N || fabsf(sum) < INFINITY)) {
    __syncthreads();
    return false;
  }
  if (n0 + lane < g.N) {
#pragma unroll 4
    for (int r = 0; r < ROWS; r++) {
      const int row = m0 + ROWS * q + r;
      if (row < g.M) put_result<THROUGH>(g, z, row, n0 + lane, row == m0 ? sum : 0.f);
    }
  }
  return true;
}

// Columns n0 .. n0 + 64 of B (K x N) summed over rows [kbeg, kend), to s[64] in LDS.  N, ldb are multiples of 4, B 16-byte aligned.
__device__ __forceinline__ void column_sums(const GemmArgs &g, int n0, int kbeg, int kend, float *__restrict__ s) {
  constexpr int U = 16;
  const int tid = threadIdx.x, group = tid >> 4, c = n0 + 4 * (tid & 15);
  const float *b = g.B + (long)kbeg * g.ldb + min(c, g.N - 4);
  const unsigned ldb = (unsigned)g.ldb;
  float4 t = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int k = kbeg + group; k < kend; k += 16 * U) {
    float4 v[U];
#pragma unroll
    for (int u = 0; u < U; u++) v[u] = *reinterpret_cast<const float4 *>(b + (size_t)(unsigned)(min(k + 16 * u, kend - 1) - kbeg) * ldb);
#pragma unroll
    for (int u = 0; u < U; u++)
      if (k + 16 * u >= kend) v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
    const float4 o = pairs(v);
    t.x += o.x, t.y += o.y, t.z += o.z, t.w += o.w;
  }
  *reinterpret_cast<float4 *>(s + 64 + tid * 4) = t;
  __syncthreads();
  if (tid < 64) {
    float v = 0.f;
#pragma unroll
    for (int p = 0; p < 16; p++) v += s[64 + p * 64 + tid];
    s[tid] = n0 + tid < g.N ? v : 0.f;
  }
  __syncthreads();
}

// two buffers of three parts
constexpr int split_lds_bytes(int BM, int BN, int BK) { return 2 * 3 * 2 * BK * (BM + BN); }

// The BM x BN tile at (m0, n0) of split `z` by the calling workgroup; S: split_lds_bytes of LDS.  FOLD: chains of
// additions end after kSplitChain of K.
template <int BM, int BN, int BK, bool TA, bool TB, bool VEC, bool FOLD, bool PULL = false, bool THROUGH = false>
__device__ __forceinline__ void split_tile(const GemmArgs &g, int m0, int n0, int z, char *__restrict__ S) {
  constexpr int WM = BM / 2, WN = BN / 2, TM = WM / 32, TN = WN / 32;
  constexpr int PA = 2 * BK * BM, PB = 2 * BK * BN, BUF = 3 * (PA + PB);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  int kbeg, kend;
  tile_k_range<BM, BN, TA, TB>(g, m0, n0, z, &kbeg, &kend);

  // (large tile: measured 3 % faster with descriptors for both operands where one of them is not k-contiguous, 4 % slower where both are)
  constexpr bool DESC = BM == 128 && BN == 128 && (TA || !TB);
  using LA = SplitLoader<BM, BK, !TA, VEC, DESC, PULL>;
  using LB = SplitLoader<BN, BK, TB, VEC, DESC>;
  LA la;
  LB lb;
  if constexpr (PULL) {
    la.prepare_pull(g, m0, tid, n0 == 0 ? g.pull_ids : nullptr);
    if (g.K <= kSameK && kend > kbeg) {
      long *one = reinterpret_cast<long *>(S);
      if (lane == 0) one[wave] = la.one;
      __syncthreads();
      const long row = one[0];
      bool same = row >= 0;
#pragma unroll
      for (int w = 1; w < 4; w++) same &= one[w] == row || one[w] == -2;
      __syncthreads();
      if (same) {
        copy_looked_up<BM, BN, BK, VEC>(g, m0, n0);
        return same_rows_product<BM, BN, VEC>(g, g.A + row, m0, n0, S);
      }
    }
  } else {
    if constexpr (!TA && !TB && !THROUGH) {
      if (g.row_ids && m0 >= g.ids_from && g.K <= kSameK && kend > kbeg && same_ids(g.row_ids, m0, min(m0 + BM, g.M)))
        return same_rows_product<BM, BN, VEC>(g, g.A + (long)m0 * g.lda, m0, n0, S);
    }
    if constexpr (!TA && TB && VEC && THROUGH) {
      if (g.row_ids && m0 >= g.ids_from && kend > kbeg && same_ids(g.row_ids, m0, min(m0 + BM, g.M)) &&
          summed_rows_product<THROUGH>(g, m0, n0, z, kbeg, kend, S))
        return;
    }
    la.prepare(g.lda, m0, g.M, tid);
  }
  // (A^T B) rows of K from `same` on, if they are equal: the sums of B's before the loops (no accumulator yet), their step behind them
  int same = kend;
  const int kall = kend;
  float one_a = 0.f, one_b = 0.f;
  if constexpr (TA && !TB && VEC && THROUGH) {
    if (g.row_ids) {
      const int from = max(kbeg, kbeg + (g.ids_from - kbeg + BK - 1) / BK * BK);
      if (from + 2 * BK <= kend && same_ids(g.row_ids, from, kend)) {
        kend = same = from;
        float *s = reinterpret_cast<float *>(S);
        column_sums(g, n0, same, kall, s);
        one_a = g.A[(long)same * g.lda + m0 + min(tid % BM, g.M - 1 - m0)];
        one_b = s[tid % BN];
        __syncthreads();
      }
    }
  }
  lb.prepare(g.ldb, n0, g.N, tid);
  const float *A = PULL ? g.A : TA ? g.A + m0 : g.A + (long)m0 * g.lda, *B = TB ? g.B + (long)n0 * g.ldb : g.B + n0;

  floatx16 acc[TM][TN], sum[FOLD ? TM : 1][FOLD ? TN : 1];
  const int nk = kend > kbeg ? (kend - kbeg + BK - 1) / BK : 0;  // steps: all, those wholly inside the range
  const int whole = kend > kbeg ? (kend - kbeg) / BK : 0;
  const int ar = wm * WM + (lane & 31), br = wn * WN + (lane & 31), half = lane >> 5;
  auto clear = [&](auto &v) {
    for (auto &row : v)
      for (floatx16 &c : row)
#pragma unroll
        for (int r = 0; r < 16; r++) c[r] = 0.f;
  };
  clear(acc);
  clear(sum);
  auto fold = [&] {
    if constexpr (FOLD) {
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
          for (int r = 0; r < 16; r++) sum[i][j][r] += acc[i][j][r];
      clear(acc);
    }
  };
  struct Regs {
    float a[LA::NU][LA::U], b[LB::NU][LB::U];
  } r0, r1;
  auto fetch = [&](Regs &r, int kt) {
    const int k0 = kbeg + kt * BK;
    if (kt < whole) {
      la.template load<true>(r.a, A, g.lda, k0, kend);
      lb.template load<true>(r.b, B, g.ldb, k0, kend);
    } else if (kt < nk) {
      la.template load<false>(r.a, A, g.lda, k0, kend);
      lb.template load<false>(r.b, B, g.ldb, k0, kend);
    }
  };
  auto put = [&](Regs &r, int kt) {
    char *to = S + (kt & 1) * BUF;
    la.store(r.a, to);
    lb.store(r.b, to + 3 * PA);
  };
  auto multiply = [&](int kt) {
    const char *SA = S + (kt & 1) * BUF, *SB = SA + 3 * PA;
#pragma unroll
    for (int s = 0; s < BK / 16; s++) {
      bf16x8 a[TM][3], b[TN][3];
#pragma unroll
      for (int p = 0; p < 3; p++) {
#pragma unroll
        for (int i = 0; i < TM; i++) a[i][p] = *reinterpret_cast<const bf16x8 *>(SA + p * PA + split_at<BK, !TA>(ar + 32 * i, 2 * s + half));
#pragma unroll
        for (int j = 0; j < TN; j++) b[j][p] = *reinterpret_cast<const bf16x8 *>(SB + p * PB + split_at<BK, TB>(br + 32 * j, 2 * s + half));
      }
      // the small products first
      constexpr int pa[6] = {2, 1, 0, 1, 0, 0}, pb[6] = {0, 1, 2, 0, 1, 0};
#pragma unroll
      for (int q = 0; q < 6; q++)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i][pa[q]], b[j][pb[q]], acc[i][j], 0, 0, 0);
    }
  };
  // step kt multiplies what is in LDS, converts step kt + 1's values, which came while step kt - 1
  // multiplied, and asks for those of step kt + 2
  if (nk > 0) {
    fetch(r0, 0);
    fetch(r1, 1);
    put(r0, 0);
  }
  __syncthreads();
  int kt = 0;
  for (; kt + 3 < whole; kt += 2) {  // every fetch in here is whole
    la.template load<true>(r0.a, A, g.lda, kbeg + (kt + 2) * BK, kend);
    lb.template load<true>(r0.b, B, g.ldb, kbeg + (kt + 2) * BK, kend);
    multiply(kt);
    put(r1, kt + 1);
    __syncthreads();
    la.template load<true>(r1.a, A, g.lda, kbeg + (kt + 3) * BK, kend);
    lb.template load<true>(r1.b, B, g.ldb, kbeg + (kt + 3) * BK, kend);
    multiply(kt + 1);
    put(r0, kt + 2);
    if (FOLD && (kt + 2) % (kSplitChain / BK) == 0) fold();
    __syncthreads();
  }
  for (; kt < nk; kt += 2) {
    fetch(r0, kt + 2);
    multiply(kt);
    if (kt + 1 < nk) put(r1, kt + 1);
    __syncthreads();
    if (kt + 1 >= nk) break;
    fetch(r1, kt + 3);
    multiply(kt + 1);
    if (kt + 2 < nk) put(r0, kt + 2);
    __syncthreads();
  }
  if constexpr (TA && !TB && VEC && THROUGH) {
    if (same < kall) {
      // A's row of 64 and the sums, as one step whose other rows of K are zero.  (An infinity meets every gradient by itself, as
      // it would have: left to unsplit_tile by the NaN it makes here.)
      constexpr int U = LA::U;
      Regs r;
#pragma unroll
      for (int i = 0; i < LA::NU; i++)
#pragma unroll
        for (int j = 0; j < U; j++) {
          const bool on = U * la.unit[i] + j == 0;
          r.a[i][j] = on ? one_a : 0.f;
          r.b[i][j] = on ? one_b : 0.f;
        }
      put(r, 0);
      __syncthreads();
      multiply(0);
      kend = kall;
    }
  }
  if constexpr (PULL) {
    if (kend > kbeg) copy_looked_up<BM, BN, BK, VEC>(g, m0, n0);
  }
  fold();
  int row = m0 + wm * WM, col = n0 + wn * WN, l = lane;
  asm volatile("" : "+v"(row), "+v"(col), "+v"(l));  // (or the addresses of the stores are kept through the loops above)
  auto finish = [&](floatx16 (&out)[TM][TN]) {
    // An infinite operand, or a finite one whose first part rounds to infinity (beyond 3.39e38), leaves
    // infinity - infinity in its parts and so NaN here, whatever the product is: the fp32 pipe decides then.
    float odd = 0.f;  // (0 times a finite number; NaN if one is not)
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) odd = fmaf(out[i][j][r], 0.f, odd);
    if (__any(!(odd == 0.f))) unsplit_tile<TM, TN, TA, TB, PULL>(g, row, col, kbeg, kend, l, out);
    store_tile<TM, TN, THROUGH>(g, out, row, col, z, l);
  };
  if constexpr (FOLD) finish(sum);
  else finish(acc);
}

// Tile `t` of a launch over row tiles [row0, row0 + rows): eight row tiles at a time, down each column
// of tiles before the next, so that the tiles an XCD runs together (consecutive t) read few panels of
// either operand.
__device__ inline void split_tile_at(int t, int row0, int rows, int tilesN, int *tm, int *tn) {
  const int band = t / (8 * tilesN), in = t - band * 8 * tilesN, high = min(8, rows - 8 * band);
  *tm = row0 + 8 * band + in % high;
  *tn = in / high;
}

template <int BM, int BN, int BK, bool TA, bool TB, bool VEC, bool FOLD, bool PULL = false>
__global__ __launch_bounds__(kThreads, BM == 128 && FOLD ? 2 : 3) void sgemm_split_kernel(GemmArgs g) {
  __shared__ __attribute__((aligned(16))) char S[split_lds_bytes(BM, BN, BK)];
  apply_live(g, TA, gridDim.y);
  const int tilesN = (g.N + BN - 1) / BN, tilesM = (g.M + BM - 1) / BM;
  if (g.live && (g.zkind == CAVS_GEMM_A_ZERO || g.zkind == CAVS_GEMM_C_UNUSED)) {
    const int inside = min(g.zrows, g.M) / BM;
    g.seg_rows = g.seg_mixed = inside < tilesM ? inside : 0;
    g.seg_cols = tilesN;
  }
  int t = blockIdx.x, row0 = 0, rows = tilesM, col0 = 0, cols = tilesN;
  if (g.seg_rows > 0) {
    for (int seg = 0;; seg++) {
      if (seg > 3) return;
      const bool inside = seg == 0 || seg == 3;
      row0 = inside ? 0 : seg == 1 ? g.seg_rows : g.seg_mixed;
      rows = (inside ? g.seg_rows : seg == 1 ? g.seg_mixed : tilesM) - row0;
      col0 = seg == 3 ? g.seg_cols : 0;
      cols = (seg == 0 ? g.seg_cols : tilesN) - col0;
      const int n = (rows * cols + 7) & ~7;
      if (t < n) {
        t = xcd_remap(t, n);
        break;
      }
      t -= n;
    }
    if (t >= rows * cols) return;
  } else if (g.live) {
    const int all = (tilesM * tilesN + 7) & ~7;
    if (t >= all) return;
    t = xcd_remap(t, all);
    if (t >= tilesM * tilesN) return;
  } else {
    t = xcd_remap(t, tilesM * tilesN);
  }
  int tm, tn;
  split_tile_at(t, row0, rows, cols, &tm, &tn);
  tn += col0;
  if constexpr (!TA && !TB) {
    if ((PULL || g.row_ids) && g.seg_rows == 0) {  // rows from both halves in turn: those of the second may be done sooner
      const int half = (tilesM + 1) / 2;
      tm = tm & 1 ? half + tm / 2 : tm / 2;
    }
  }
  split_tile<BM, BN, BK, TA, TB, VEC, FOLD, PULL>(g, tm * BM, tn * BN, blockIdx.y, S);
}

}  // namespace cavs
