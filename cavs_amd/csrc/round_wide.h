// Tiles of sixteen rows for the launches that keep several rounds resident (round_group.h): the same fp32
// products as the four-row tiles, four times the rows per pass.
//
// A list of a few rows is bound by latency, and tiles of four rows are the shortest way through it.  A list of
// many rows is bound by what a tile costs.  At H = 512, Tree-LSTM, the fp32 MFMAs of four rows are 1280 cycles of a
// SIMD's matrix pipe, but a tile takes 2580 forward and 2750 backward: behind them come the sums over the four k slots (64
// vector instructions a wavefront) and operand fetches that give every quad of lanes four cache lines to
// collect.  On the 16 x 16 x 4 shape there are no slots, and a row's operands come as four lanes x 16 consecutive
// bytes; they cross to the lanes the MFMA wants them in (row l % 16, k slot l / 16) through LDS, in memory of the
// wavefront's own: no barrier.  Positions are permuted by the row so that no bank is hit twice (4.25 cycles a read
// where permuting by row / 4 takes 8).  Sixteen rows take 6700 cycles forward, 7000 backward, of which 5120 are MFMAs.
// The weights are those the four-row tiles keep in registers, so a list chooses tile by tile.
//   64 trees, H = 512: 15 lists a group of 62, 35, 21, 12 .. 1 rows, 72.6 us forward and 82.1 backward -> 68.6 / 78.4
//   64 trees, H = 256, Tree-FC: 45.6 / 40.1 -> 39.1 / 35.6
//   128 chains, H = 512, 100 rounds of up to 16 rows a group: 399 / 490 -> 388 / 430
#pragma once
#include "round_sync.h"

namespace cavs {

// Rows past the last whole tile of sixteen that are still worth one.  (Eight rows are two tiles of four.)
constexpr int kWideRest = 9;
__device__ inline int wide_tiles(int n) { return (n + 16 - kWideRest) >> 4; }

// The lane's place among the 64 float4 that sixteen k of sixteen rows take in the staging memory
__device__ inline int wide_put(int lane) { return (lane & ~3) + ((lane & 3) ^ ((lane >> 3) & 3)); }       // row lane / 4, k 4 (lane % 4)
__device__ inline int wide_get(int lane) { return 4 * (lane & 15) + ((lane >> 4) ^ ((lane >> 1) & 3)); }  // row lane % 16, k 4 (lane / 16)

// Sums of tile t of NP products over the wavefront's k: [tile][wavefront][product][lane][4 rows], in the memory of
// the four four-row tiles it stands for
template <int NP>
__device__ inline void wide_park(float *red, const floatx4 (&acc)[NP], int t, int ks, int lane) {
#pragma unroll
  for (int p = 0; p < NP; p++) *reinterpret_cast<floatx4 *>(red + ((t * 8 + ks) * NP + p) * 256 + lane * 4) = acc[p];
}
// product p of row 4 ks + lane / 16 of the list, column lane % 16, added up in wavefront order
template <int NP>
__device__ inline void wide_sum(const float *red, int ks, int lane, float (&v)[NP]) {
  const float *pre = red + (ks >> 2) * 8 * NP * 256 + ((ks & 3) * 16 + (lane & 15)) * 4 + (lane >> 4);
#pragma unroll
  for (int p = 0; p < NP; p++) {
    float s = 0.f;
#pragma unroll
    for (int g = 0; g < 8; g++) s += pre[(g * NP + p) * 256];
    v[p] = s;
  }
}
// what a launch parks: 32 rows of sixteen columns, eight wavefronts, NP products
constexpr size_t group_red_bytes(int NP) { return (size_t)8 * 32 * 16 * NP * sizeof(float); }

// ------------------------------------------------------------------ forward
template <int MODEL, int GPW>
struct WideFwd {
  static constexpr int NP = MODEL == GROUP_TREELSTM ? 5 : MODEL == GROUP_LSTM ? 4 : 2, NW = MODEL == GROUP_TREEFC ? 2 : 4;
  static constexpr int NC = MODEL == GROUP_LSTM ? 1 : 2;
  static constexpr size_t kLds = group_red_bytes(NP) + (size_t)8 * NC * GPW * 64 * sizeof(float4);
  float4 v[NC][GPW];  // the rows of the tile to come
  bool on[NC];
  int ks, lane, groups;  // k-groups of sixteen: ks * GPW .. + groups
  float4 *stage;

  __device__ inline WideFwd(const GroupFwdArgs &a, int ks_, int lane_, float *red) : ks(ks_), lane(lane_) {
    groups = min(GPW, max(0, a.H / 16 - ks * GPW));
    stage = reinterpret_cast<float4 *>(red + group_red_bytes(NP) / sizeof(float)) + ks * (NC * GPW * 64);
  }
  // the rows of tile t of a list of n on their way (rows past the list's end stand for its last; a missing child
  // reads weights; k-groups beyond H read the first and drop it)
  __device__ inline void fetch(const GroupFwdArgs &a, const int4 *rt, int n, int t, long MW) {
    const int i = 16 * t + (lane >> 2);
    const int4 c = rt[2 * (i < n ? i : n - 1)];
#pragma unroll
    for (int s = 0; s < NC; s++) {
      const int row = s == 0 ? c.y : c.z;
      on[s] = row >= 0;
      const float *p = (row >= 0 ? a.pool + row * MW : a.Wp) + 4 * (lane & 3);
#pragma unroll
      for (int g = 0; g < GPW; g++) v[s][g] = ld4(p + (g < groups ? 16 * (ks * GPW + g) : 0));
    }
  }
  // tile t, whose rows have been asked for; then those of tile t + 1 where there is one.  Nothing here is conditional but
  // that: the waits come out exact.
  __device__ inline void tile(const GroupFwdArgs &a, const int4 *rt, int n, int t, bool more, long MW, const float4 (&wt)[NW][GPW], float *red) {
    float4 *to = stage + wide_put(lane);
    const float4 *from = stage + wide_get(lane);
#pragma unroll
    for (int s = 0; s < NC; s++)
#pragma unroll
      for (int g = 0; g < GPW; g++) to[(s * GPW + g) * 64] = sel4(on[s] && g < groups, v[s][g]);
    if (more) fetch(a, rt, n, t + 1, MW);
    __builtin_amdgcn_wave_barrier();
    float4 f[NC][GPW];
#pragma unroll
    for (int g = 0; g < GPW; g++)
#pragma unroll
      for (int s = 0; s < NC; s++) f[s][g] = from[(s * GPW + g) * 64];
    floatx4 acc[NP];
#pragma unroll
    for (int p = 0; p < NP; p++) acc[p] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int g = 0; g < GPW; g++) {
      const float4 &A = f[0][g], &B = f[NC - 1][g];
      const float4 S = make_float4(A.x + B.x, A.y + B.y, A.z + B.z, A.w + B.w);
#pragma unroll
      for (int c = 0; c < 4; c++) {
        if constexpr (MODEL == GROUP_TREELSTM) {
          acc[0] = Mma<16>::mma(elem(S, c), elem(wt[0][g], c), acc[0]);
          acc[1] = Mma<16>::mma(elem(S, c), elem(wt[1][g], c), acc[1]);
          acc[2] = Mma<16>::mma(elem(S, c), elem(wt[2][g], c), acc[2]);
          acc[3] = Mma<16>::mma(elem(A, c), elem(wt[3][g], c), acc[3]);
          acc[4 % NP] = Mma<16>::mma(elem(B, c), elem(wt[3][g], c), acc[4 % NP]);
        } else if constexpr (MODEL == GROUP_LSTM) {
#pragma unroll
          for (int q = 0; q < 4; q++) acc[q % NP] = Mma<16>::mma(elem(A, c), elem(wt[q % NW][g], c), acc[q % NP]);
        } else {
          acc[0] = Mma<16>::mma(elem(A, c), elem(wt[0][g], c), acc[0]);
          acc[1] = Mma<16>::mma(elem(B, c), elem(wt[1][g], c), acc[1]);
        }
      }
    }
    wide_park<NP>(red, acc, t, ks, lane);
  }
};

// ------------------------------------------------------------------ backward
template <int MODEL, int GPW>
struct WideBwd {
  static constexpr int NP = MODEL == GROUP_TREELSTM ? 3 : MODEL == GROUP_LSTM ? 1 : 2;
  // k-groups of the product over a row of dA (K = 3H, 4H, H) and of those over the rows of dF; a tile takes its U
  // k-groups D at a time (five of the twenty at H = 512: ten spill)
  static constexpr int KL = MODEL == GROUP_TREELSTM ? 3 * GPW : MODEL == GROUP_LSTM ? 4 * GPW : GPW, KF = MODEL == GROUP_TREELSTM ? GPW : 0;
  static constexpr int U = KL + 2 * KF, D = U <= 10 ? U : U > 16 && U % 4 == 0 ? U / 4 : U % 2 == 0 ? U / 2 : U / 3;
  static_assert(U % D == 0, "a tile is whole turns");
  static constexpr int NS = MODEL == GROUP_LSTM ? 1 : GPW;
  static constexpr size_t kLds = group_red_bytes(NP) + (size_t)8 * (D * 64 + 1) * sizeof(float4);
  float4 v[D];
  int ks, lane, gl, gf;  // k-groups of dA this wavefront has, and of dF
  float4 *stage, *none;  // its rows on their way, and zeros

  __device__ inline WideBwd(const GroupBwdArgs &a, int ks_, int lane_, float *red) : ks(ks_), lane(lane_) {
    const int KG = a.H / 16;
    gl = min(KL, max(0, KL / GPW * KG - ks * KL));
    gf = min(GPW, max(0, KG - ks * GPW));
    stage = reinterpret_cast<float4 *>(red + group_red_bytes(NP) / sizeof(float)) + ks * (D * 64);
    none = reinterpret_cast<float4 *>(red + group_red_bytes(NP) / sizeof(float)) + 8 * (D * 64) + ks;
  }
  __device__ inline void clear() { *none = zero4(); }  // (before the launch's first barrier)
  struct Row {
    const float *l, *f;
  };
  // where this lane reads the row of tile t it fetches (rows past the list's end stand for its first; their results are not written)
  __device__ inline Row row(const GroupBwdArgs &a, const int4 *rt, int n, int t) const {
    const int i = 16 * t + (lane >> 2);
    const long r = rt[2 * (i < n ? i : 0)].x;
    return {a.dA + r * a.ld + 4 * (lane & 3), MODEL == GROUP_TREELSTM ? a.dF + 2 * r * a.H + 4 * (lane & 3) : nullptr};
  }
  // k-groups u0 .. of the row (those beyond the product's K read its first, and zeros stand for them in the product: their weights are
  // zero, but zero times an infinity is a NaN.  The address is chosen, when a fragment is read: a branch around stores of zeros
  // stands before the waits for the loads to come.  The launch of 64 trees, H = 512: 80.5 us so, 84.5 behind a branch and 79.5 with
  // nothing dropped; Tree-FC, H = 256: 36.7 and 36.4, 39.3 with the value masked)
  __device__ inline void fetch(const GroupBwdArgs &a, const Row &r, int u0) {
#pragma unroll
    for (int i = 0; i < D; i++) {
      const int u = u0 + i;
      if (u < KL) {
        v[i] = ld4(r.l + (u < gl ? 16 * (ks * KL + u) : 0));
      } else {
        const int g = (u - KL) % (KF ? KF : 1);
        v[i] = ld4(r.f + (u < KL + KF ? 0 : a.H) + (g < gf ? 16 * (ks * GPW + g) : 0));
      }
    }
  }
  __device__ inline void start(const GroupBwdArgs &a, const int4 *rt, int n) { fetch(a, row(a, rt, n, 0), 0); }
  __device__ inline void tile(const GroupBwdArgs &a, const int4 *rt, int n, int t, bool more, const float4 (&wl)[KL], const float4 (&ws)[NS],
                              float *red) {
    floatx4 acc[NP], two = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int p = 0; p < NP; p++) acc[p] = floatx4{0.f, 0.f, 0.f, 0.f};
    const Row now = row(a, rt, n, t);
    float4 *to = stage + wide_put(lane);
    const float4 *from = stage + wide_get(lane);
#pragma unroll
    for (int u0 = 0; u0 < U; u0 += D) {
#pragma unroll
      for (int i = 0; i < D; i++) to[i * 64] = v[i];
      if (u0 + D < U) fetch(a, now, u0 + D);
      else if (more) fetch(a, row(a, rt, n, t + 1), 0);
      __builtin_amdgcn_wave_barrier();
      float4 f[D];
#pragma unroll
      for (int i = 0; i < D; i++) {
        const int u = u0 + i;
        f[i] = *((u < KL ? u < gl : (u - KL) % (KF ? KF : 1) < gf) ? from + i * 64 : none);
      }
#pragma unroll
      for (int i = 0; i < D; i++) {
        const int u = u0 + i;
        const float4 &x = f[i];
#pragma unroll
        for (int c = 0; c < 4; c++) {
          if constexpr (MODEL == GROUP_TREEFC) {
            acc[0] = Mma<16>::mma(elem(x, c), elem(wl[u % KL], c), acc[0]);
            acc[NP - 1] = Mma<16>::mma(elem(x, c), elem(ws[u % NS], c), acc[NP - 1]);
          } else if (u < KL) {  // (in two accumulators: each MFMA would wait for the one before otherwise)
            if (c & 1) two = Mma<16>::mma(elem(x, c), elem(wl[u % KL], c), two);
            else acc[0] = Mma<16>::mma(elem(x, c), elem(wl[u % KL], c), acc[0]);
          } else {
            const int s = u < KL + KF ? 1 : 2;
            acc[s % NP] = Mma<16>::mma(elem(x, c), elem(ws[(u - KL) % (KF ? KF : 1)], c), acc[s % NP]);
          }
        }
      }
    }
    if constexpr (MODEL != GROUP_TREEFC) {
#pragma unroll
      for (int r = 0; r < 4; r++) acc[0][r] += two[r];
    }
    wide_park<NP>(red, acc, t, ks, lane);
  }
};

}  // namespace cavs
