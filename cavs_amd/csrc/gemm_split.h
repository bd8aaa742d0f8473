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
// PULL (k-contiguous): rows are looked up (GemmArgs::pull_*), and those a workgroup reads go on into pull_copy.
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
  bool in[PULL ? NU : 1];       // the row is inside the operand and has an id
  float *copy[PULL ? NU : 1];  // where the unit goes as well, or nullptr
  int copy_mod = 1, copy_rem = 0;
  __device__ inline void prepare_pull(const GemmArgs &g, int x0, int tid, float *ids_out, int mod, int rem) {
    static_assert(!PULL || KC, "looked-up rows are k-contiguous");
    copy_mod = mod;
    copy_rem = rem;
#pragma unroll
    for (int i = 0; i < NU; i++) {
      const int u = tid + kThreads * i, x = u / PER, gx = x0 + x;
      unit[i] = u % PER;
      at[i] = split_at<BK, KC>(x, unit[i] >> 1) + 8 * (unit[i] & 1);
      long off = -1;
      if (gx < g.M) {
        const float id = g.pull_x[g.pull_rows[gx]];
        off = (long)(int)(id * (float)g.K);
        if (ids_out && unit[i] == 0) ids_out[gx] = id;
      }
      in[i] = off >= 0;
      boff[i] = 4 * ((Off)(in[i] ? off : 0) + U * unit[i]);
      copy[i] = gx < g.M ? g.pull_copy + (long)gx * g.ld_copy + U * unit[i] : nullptr;
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
        if constexpr (PULL) {
          const int left = in[i] ? kend - k0 - U * unit[i] : 0;
          if constexpr (VEC) {  // (K is a multiple of 4)
            float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
            if (left > 0) a = *reinterpret_cast<const float4 *>(q);
            v[i][0] = a.x, v[i][1] = a.y, v[i][2] = a.z, v[i][3] = a.w;
          } else {
#pragma unroll
            for (int j = 0; j < U; j++) v[i][j] = j < left ? q[j] : 0.f;
          }
          if (copy[i] && (k0 / BK) % copy_mod == copy_rem) {
            const int room = kend - k0 - U * unit[i];
            if constexpr (VEC) {
              if (room > 0) *reinterpret_cast<float4 *>(copy[i] + k0) = make_float4(v[i][0], v[i][1], v[i][2], v[i][3]);
            } else {
#pragma unroll
              for (int j = 0; j < U; j++)
                if (j < room) copy[i][k0 + j] = v[i][j];
            }
          }
        } else if constexpr (WHOLE && VEC) {
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

  __device__ inline void store(const float (&v)[NU][U], char *__restrict__ S) const {
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
    // the column tiles of this row tile that do run share the copying
    const int tilesN = (g.N + BN - 1) / BN, tn = n0 / BN;
    const int active = (g.zkind == CAVS_GEMM_C_UNUSED && m0 + BM <= g.zrows) ? min(tilesN, (g.zcol + BN - 1) / BN) : tilesN;
    la.prepare_pull(g, m0, tid, n0 == 0 ? g.pull_ids : nullptr, active, tn);
  } else {
    la.prepare(g.lda, m0, g.M, tid);
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
  auto put = [&](const Regs &r, int kt) {
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
    const int inside = min(g.zrows, g.M) / BM * tilesN;
    g.zseg = inside < tilesM * tilesN ? inside : 0;
  }
  int t, row0 = 0, rows = tilesM;
  if (g.zseg > 0) {
    const int first = (g.zseg + 7) & ~7, rest = (tilesM * tilesN - g.zseg + 7) & ~7, b = blockIdx.x;
    if (b >= first + rest) return;
    if (b < first) {
      t = xcd_remap(b, first);
      rows = g.zseg / tilesN;
    } else {
      t = xcd_remap(b - first, rest);
      row0 = g.zseg / tilesN;
      rows = tilesM - row0;
    }
    if (t >= rows * tilesN) return;
  } else if (g.live) {
    const int all = (tilesM * tilesN + 7) & ~7;
    if ((int)blockIdx.x >= all) return;
    t = xcd_remap(blockIdx.x, all);
    if (t >= tilesM * tilesN) return;
  } else {
    t = xcd_remap(blockIdx.x, tilesM * tilesN);
  }
  int tm, tn;
  split_tile_at(t, row0, rows, tilesN, &tm, &tn);
  split_tile<BM, BN, BK, TA, TB, VEC, FOLD, PULL>(g, tm * BM, tn * BN, blockIdx.y, S);
}

}  // namespace cavs
