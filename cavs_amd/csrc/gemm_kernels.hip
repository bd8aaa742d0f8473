// fp32 products for the gate products of the vertex functions, row-major: NN (X*W), NT (dY*W^T) and
// TN (X^T*dY), on the bf16 matrix pipe at full fp32 precision (gemm_split.h): tiles of 128 x 128 for
// problems that fill the chip, 64 x 64 otherwise.
// Workgroup ids are remapped so that consecutive tiles (which share operand panels)
// run on the same XCD and hit the same L2.  Products with too few tiles to fill the
// chip take one of two other routes: skinny ones (the tail rounds of a batch) a
// kernel whose wavefronts split K inside the workgroup, tall-K ones (the deferred
// weight gradients) split K over workgroups with the partials reduced in a fixed
// order by a second kernel.
#include <algorithm>
#include <type_traits>

#include <atomic>

#include "bench_probes.h"
#include "colsum_common.h"
#include "common.h"
#include "embed_common.h"
#include "gemm_common.h"
#include "gemm_split.h"

namespace cavs {

// Several independent products in one launch (the deferred weight gradients of a step and the
// embedding gradient's product): alone, each of them is a single round of workgroups that all
// load, multiply and store at the same time; together their phases overlap and the chip sees
// one long launch.  Workgroup b belongs to product p with first[p] <= b < first[p+1] (each
// product's share is padded to a multiple of 8, so that b % 8 is the XCD within the share as
// well); within the share, tile = local % tiles[p] and K split = local / tiles[p].
constexpr int kGroupMax = 8;
struct GemmGroup {
  GemmArgs g[kGroupMax];
  int first[kGroupMax + 1];
  int tiles[kGroupMax];
  int splits[kGroupMax];
  int form[kGroupMax];  // transA * 2 + transB
  // Tiles and splits whose rows may be all one (GemmArgs::row_ids): those behind the first long_tiles, long_splits.  They are done soon, so
  // they come behind everything else (from after[p] on) and are dealt to the XCDs by themselves: among the others they left some XCDs
  // without work.
  int long_tiles[kGroupMax], long_splits[kGroupMax], after[kGroupMax + 1];
  int count;
};

// The embedding gradient behind one product of a group (cavs_sgemm_group_embed_bwd): the rows of
// that product's result are scatter-added into the table by extra workgroups of the launch that
// reduces the other products' K splits, reading the product's own partials directly.
struct EmbedTail {
  float *dtable;
  const float *ids;
  const float *dy;   // the result, or the first of `parts` partial results `part_stride` floats apart
  long ld_dy, part_stride;
  int parts;
  float *copy;       // where the summed result goes as well (the product's C) when parts > 1
  long ld_copy;
  int n, E, gx;      // gx row chunks of 64
  const int *live;   // cavs_gemm_desc::live of the product
};

// What a group's launch finishes by itself where it has counters: the workgroup that arrives last at a tile of a product whose K
// is split adds up the tile's partial sums, in the order of the splits whoever is last, and scatters the tile of the
// product that feeds the embedding's gradient.  Partial sums go past the L2 (THROUGH), and the count behind
// them; the last one puts the counter back to zero.  Column sums come along as workgroups behind the products'.
// As launches of their own these were latency, not work -- ids, parts and atomic adds one behind the other, 4.5 us between
// two launches.  What bounds the end of the launch now are those trips: so all parts of a tile are in flight at once (one
// after the other: 24.6 us where it takes 19.6), and the ids are looked up in front of the product.
//   us, products + reduction (+ scatter) (+ column sums) -> one launch, gaps not counted
//   64 trees, H = 512 (2370 vertices): 74.0 + 15.6 -> 77.9        25 trees, H = 150: 15.6 + 13.4 -> 19.9
//   16 chains of 20, H = 128, 1000 classes: 11.9 + 4.1 + 6.1 and 11.9 + 12.0 + 6.1 -> 27.3 together
struct GroupFold {
  int *counters;          // one per tile of a split product, zero; null: a launch behind this one adds up
  int first[kGroupMax];   // the product's first
  int embed;              // product whose tiles are scattered, or -1
  EmbedTail tail;
  ColsumParts sums;       // chunks > 0: its column sums by the workgroups behind the products'
};

// the partial sums of tile (m0, n0) of a product added up; thread: column lane of rows 16 wave ..
__device__ inline void fold_tile(const GemmArgs &g, int splits, int m0, int n0) {
  const int lane = threadIdx.x & 63, row0 = __builtin_amdgcn_readfirstlane(m0 + 16 * (threadIdx.x >> 6)), c = n0 + lane;
  if (row0 >= g.M || c >= g.N) return;
  const long stride = (long)g.M * g.N;
  float acc[16];
#pragma unroll
  for (int u = 0; u < 16; u++) acc[u] = 0.f;
  const ThroughRows rows{g.N, g.M - 1 - row0, 4 * c};
  const float *p = g.ws + (long)row0 * g.N;
  for (int z = 0; z < splits; z += 4, p += 4 * stride) {  // four parts in flight: one at a time, each is a trip to memory
    float v[4][16];
#pragma unroll
    for (int k = 0; k < 4; k++) rows.load(p + (z + k < splits ? k : 0) * stride, v[k]);
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if (z + k >= splits) break;
#pragma unroll
      for (int u = 0; u < 16; u++) acc[u] += v[k][u];
    }
  }
#pragma unroll
  for (int u = 0; u < 16; u++) {
    if (row0 + u >= g.M) continue;
    float *to = g.C + (row0 + u) * g.ldc + c;
    float v = g.alpha * acc[u];
    if (g.beta != 0.f) v += g.beta * *to;
    *to = v;
  }
}

template <bool VEC>
__global__ __launch_bounds__(kThreads, 4) void sgemm_group_kernel(GemmGroup G, GroupFold F) {
  constexpr int BM = 64, BN = 64, BK = 16;
  __shared__ __attribute__((aligned(16))) char S[split_lds_bytes(BM, BN, BK)];
  const int end = G.first[G.count] + G.after[G.count];
  if ((int)blockIdx.x >= end) {
    const int b = blockIdx.x - end, across = (F.sums.w + 63) / 64;
    return colsum_part_block(F.sums, b % across, b / across, reinterpret_cast<float(*)[64]>(S));
  }
  const bool soon = (int)blockIdx.x >= G.first[G.count];
  int local = blockIdx.x, p = 0;
  if (soon) {
    local -= G.first[G.count];
    while (p + 1 < G.count && local >= G.after[p + 1]) p++;
    local -= G.after[p];
  } else {
    while (p + 1 < G.count && local >= G.first[p + 1]) p++;
    local -= G.first[p];
  }
  GemmArgs g = G.g[p];
  apply_live(g, G.form[p] >= 2, G.splits[p]);
  const int tiles = g.live ? (g.M + BM - 1) / BM * ((g.N + BN - 1) / BN) : G.tiles[p];
  const int longT = g.live ? tiles : G.long_tiles[p], longZ = G.long_splits[p];
  const int share = soon ? tiles * G.splits[p] - longT * longZ : longT * longZ, padded = (share + 7) & ~7;
  if (local >= padded) return;
  const int w = xcd_remap(local, padded);
  if (w >= share) return;
  int t = w % longT, z = w / longT;
  if (soon) {
    const bool rows = longT < tiles;
    const int across = rows ? tiles - longT : tiles;
    t = (rows ? longT : 0) + w % across;
    z = (rows ? 0 : longZ) + w / across;
  }
  const int tilesN = (g.N + BN - 1) / BN, m0 = t / tilesN * BM, n0 = t % tilesN * BN;
  int mine = -1;  // (asked for in front of the product, looked at behind it)
  if (F.counters && F.embed == p && m0 < min(F.tail.n, g.M)) mine = embed_row(F.tail.ids, min(F.tail.n, g.M), F.tail.E, m0 / kEmbedRows);
  switch (G.form[p]) {
    case 0: split_tile<BM, BN, BK, false, false, VEC, true, false, true>(g, m0, n0, z, S); break;
    case 1: split_tile<BM, BN, BK, false, true, VEC, true, false, true>(g, m0, n0, z, S); break;
    case 2: split_tile<BM, BN, BK, true, false, VEC, true, false, true>(g, m0, n0, z, S); break;
    default: split_tile<BM, BN, BK, true, true, VEC, true, false, true>(g, m0, n0, z, S); break;
  }
  if (!F.counters) return;
  asm volatile("" : "+s"(p), "+s"(t));  // (what follows reads its sizes again: kept over the product they cost registers)
  const int splits = G.splits[p];
  const bool scatter = F.embed == p;
  if (splits == 1 && !scatter) return;
  EmbedHot hot{0, false};
  if (scatter) hot = embed_hot(mine);  // while the stores are on their way
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this workgroup's part of the tile has arrived
  __syncthreads();
  if (splits > 1) {
    int *count = F.counters + F.first[p] + t, *last = reinterpret_cast<int *>(S);
    if (threadIdx.x == 0) *last = __hip_atomic_fetch_add(count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (*last != splits - 1) return;
    if (threadIdx.x == 0) __hip_atomic_store(count, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  GemmArgs h = G.g[p];
  apply_live(h, G.form[p] >= 2, splits);
  const int across = (h.N + BN - 1) / BN, tm = t / across, tn = t % across;
  if (!scatter) return fold_tile(h, splits, tm * BM, tn * BN);
  const EmbedTail &e = F.tail;
  const int n = min(e.n, h.M);
  if (tm * BM >= n) return;
  embed_bwd_rows<true>(e.dtable, mine, [&] { return hot; }, e.dy, e.ld_dy, e.parts, (long)h.M * h.N, e.copy, e.ld_copy, n, e.E, tm, tn);
}
static_assert(kEmbedRows == 64 && kEmbedCols == 64, "a tile of a group is a block of the scatter-add");

// p[0] + p[stride] + ... in that order, four loads in flight at a time (one at a time, a reduction over
// four splits was four trips to memory in a row)
__device__ inline float sum_splits(const float *__restrict__ p, int splits, long stride) {
  float acc = 0.f;
  for (int z = 0; z < splits; z += 4) {
    float v[4];
#pragma unroll
    for (int k = 0; k < 4; k++) v[k] = z + k < splits ? p[(long)(z + k) * stride] : 0.f;
#pragma unroll
    for (int k = 0; k < 4; k++) acc += v[k];
  }
  return acc;
}

// the split products of a group, reduced in one launch (same fixed order as splitk_reduce_kernel)
__global__ void splitk_reduce_group_kernel(GemmGroup R) {
  // first[] counts 256-thread workgroups per product here
  int p = 0;
  while (p + 1 < R.count && (int)blockIdx.x >= R.first[p + 1]) p++;
  GemmArgs g = R.g[p];
  apply_live(g, R.form[p] >= 2, R.splits[p]);
  const int splits = R.splits[p];
  long idx = (long)(blockIdx.x - R.first[p]) * blockDim.x + threadIdx.x;
  long total = (long)g.M * g.N;
  if (idx >= total) return;
  const float acc = sum_splits(g.ws + idx, splits, total);
  int r = (int)(idx / g.N), c = (int)(idx % g.N);
  float v = g.alpha * acc;
  if (g.beta != 0.f) v += g.beta * g.C[r * g.ldc + c];
  if (g.D) v += g.D[(long)(r >> g.dshift) * g.ldd + c];
  g.C[r * g.ldc + c] = v;
}

// What the matrix pipes sustain with nothing else in the way (cavs_mfma_probe): every wavefront
// issues `iters` rounds of eight independent 32x32x2 MFMAs on operands it keeps in registers.
__global__ __launch_bounds__(256) void mfma_probe_kernel(float *__restrict__ out, int iters) {
  floatx16 acc[8];
#pragma unroll
  for (int i = 0; i < 8; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) acc[i][r] = 0.f;
  const float a = 1.f + (threadIdx.x & 7) * 0.125f, b = 0.5f - (threadIdx.x & 3) * 0.0625f;
  for (int it = 0; it < iters; it++) {
#pragma unroll
    for (int i = 0; i < 8; i++) acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc[i], 0, 0, 0);
  }
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 8; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) s += acc[i][r];
  out[(long)blockIdx.x * blockDim.x + threadIdx.x] = s;
}

__global__ __launch_bounds__(256) void splitk_reduce_group_embed_kernel(GemmGroup R, EmbedTail e) {
  const int nred = R.first[R.count];
  if ((int)blockIdx.x >= nred) {
    const int vb = blockIdx.x - nred;
    if (e.live) {
      e.n = min(e.n, e.live[0]);
      if (e.parts > 1) e.part_stride = (long)e.n * e.ld_dy;
      if (vb % e.gx * kEmbedRows >= e.n) return;
    }
    embed_bwd_block(e.dtable, e.ids, e.dy, e.ld_dy, e.parts, e.part_stride, e.copy, e.ld_copy, e.n, e.E, vb % e.gx, vb / e.gx);
    return;
  }
  int p = 0;
  while (p + 1 < R.count && (int)blockIdx.x >= R.first[p + 1]) p++;
  GemmArgs g = R.g[p];
  apply_live(g, R.form[p] >= 2, R.splits[p]);
  const int splits = R.splits[p];
  long idx = (long)(blockIdx.x - R.first[p]) * blockDim.x + threadIdx.x;
  long total = (long)g.M * g.N;
  if (idx >= total) return;
  const float acc = sum_splits(g.ws + idx, splits, total);
  int r = (int)(idx / g.N), c = (int)(idx % g.N);
  float v = g.alpha * acc;
  if (g.beta != 0.f) v += g.beta * g.C[r * g.ldc + c];
  g.C[r * g.ldc + c] = v;
}

// C = alpha * sum_z ws[z] + beta * C (+ D rows), z ascending: a fixed order, so the
// result does not depend on how the workgroups were scheduled.
__global__ void splitk_reduce_kernel(GemmArgs g, int splits, bool tA) {
  apply_live(g, tA, splits);
  long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  long total = (long)g.M * g.N;
  if (idx >= total) return;
  const float acc = sum_splits(g.ws + idx, splits, total);
  int r = (int)(idx / g.N), c = (int)(idx % g.N);
  float v = g.alpha * acc;
  if (g.beta != 0.f) v += g.beta * g.C[r * g.ldc + c];
  if (g.D) v += g.D[(long)(r >> g.dshift) * g.ldd + c];
  g.C[r * g.ldc + c] = v;
}

// Skinny products (few rows: the tail rounds of a batch).  Such a product is a
// latency chain, not a throughput problem: the weights must stream past a handful of
// rows.  One workgroup owns a (32*TM) x 32 tile of C and its W wavefronts split K
// between them; every wavefront feeds the MFMA straight from global memory (the B
// operand of a 32x32x2 step is 32 consecutive floats per half-wave, so no LDS staging
// is needed) with several k-groups in flight, and the W partial tiles are summed
// through LDS in wavefront order (deterministic).  Bound by its trips to memory one behind the other, three of them before a looked-up
// row's first values: B's are under way before them, and the partial tiles are parked side by side and added by all threads (in place, a
// wavefront after the other, was a barrier each): 31 looked-up rows of 300, 2048 columns, 10.4 -> 9.5 us.  A is [M,K] row-major; B is [K,N]
// (TB = false) or [N,K] (TB = true).  Needs K, lda (and ldb when TB) multiples of 4.
template <int TM, bool TB, int W>
__global__ __launch_bounds__(W * 64) void sgemm_skinny_kernel(GemmArgs g) {
  constexpr int U = 4;  // k-groups of 8 in flight
  __shared__ float red[W][TM * 16 * 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int j = lane & 31, h = lane >> 5;
  const int n0 = blockIdx.x * 32, m0 = blockIdx.y * 32 * TM;
  const int kper = ((g.K + W - 1) / W + 7) / 8 * 8;
  const int kb = wave * kper, ke = min(g.K, kb + kper);
  const bool col_ok = n0 + j < g.N;
  auto fetch_b = [&](int k0, float (&b)[U][4]) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int kk = k0 + 8 * u + 4 * h;
      if constexpr (TB) {
        float4 q = (kk < ke && col_ok) ? *reinterpret_cast<const float4 *>(g.B + (long)(n0 + j) * g.ldb + kk)
                                       : make_float4(0.f, 0.f, 0.f, 0.f);
        b[u][0] = q.x; b[u][1] = q.y; b[u][2] = q.z; b[u][3] = q.w;
      } else {
#pragma unroll
        for (int c = 0; c < 4; c++)
          b[u][c] = (col_ok && kk + c < ke) ? g.B[(long)(kk + c) * g.ldb + n0 + j] : 0.f;
      }
    }
  };
  float4 a0[U][TM], a1[U][TM];
  float b0[U][4], b1[U][4];
  if (kb < ke) fetch_b(kb, b0);
  // where row m0 + 32 t + j of A is, in floats from g.A (-1: a zero row); looked-up rows (GemmArgs::pull_*)
  // go on into pull_copy, a wavefront's k range per column tile
  long arow[TM];
  const bool pulls = g.pull_rows != nullptr;
  const bool copies = pulls && (int)(wave % gridDim.x) == (int)blockIdx.x;
#pragma unroll
  for (int t = 0; t < TM; t++) {
    const int row = m0 + 32 * t + j;
    arow[t] = row < g.M ? (long)row * g.lda : -1;
    if (pulls && row < g.M) {
      const float id = g.pull_x[g.pull_rows[row]];
      arow[t] = (long)(int)(id * (float)g.K);
      if (blockIdx.x == 0 && wave == 0 && h == 0) g.pull_ids[row] = id;
    }
  }

  floatx16 acc[TM];
#pragma unroll
  for (int t = 0; t < TM; t++)
#pragma unroll
    for (int r = 0; r < 16; r++) acc[t][r] = 0.f;

  // one stage = U groups of 8 k values; the next stage's operands are fetched before
  // the MFMAs of the current one are issued, so memory latency overlaps the matrix pipe
  auto fetch_a = [&](int k0, float4 (&a)[U][TM]) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int kk = k0 + 8 * u + 4 * h;
      const bool kin = kk < ke;
#pragma unroll
      for (int t = 0; t < TM; t++) {
        a[u][t] = (kin && arow[t] >= 0) ? *reinterpret_cast<const float4 *>(g.A + arow[t] + kk) : make_float4(0.f, 0.f, 0.f, 0.f);
        if (copies && kin) {
          const int row = m0 + 32 * t + j;
          if (row < g.M) *reinterpret_cast<float4 *>(g.pull_copy + (long)row * g.ld_copy + kk) = a[u][t];
        }
      }
    }
  };
  auto multiply = [&](const float4 (&a)[U][TM], const float (&b)[U][4]) {
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int t = 0; t < TM; t++) {
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[u][t].x, b[u][0], acc[t], 0, 0, 0);
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[u][t].y, b[u][1], acc[t], 0, 0, 0);
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[u][t].z, b[u][2], acc[t], 0, 0, 0);
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[u][t].w, b[u][3], acc[t], 0, 0, 0);
      }
  };
  constexpr int S = 8 * U;
  if (kb < ke) fetch_a(kb, a0);
  for (int k0 = kb; k0 < ke; k0 += 2 * S) {
    if (k0 + S < ke) {
      fetch_b(k0 + S, b1);
      fetch_a(k0 + S, a1);
    }
    multiply(a0, b0);
    if (k0 + S < ke) {
      if (k0 + 2 * S < ke) {
        fetch_b(k0 + 2 * S, b0);
        fetch_a(k0 + 2 * S, a0);
      }
      multiply(a1, b1);
    }
  }

  // the W partial tiles, added up in wavefront order
#pragma unroll
  for (int t = 0; t < TM; t++)
#pragma unroll
    for (int r = 0; r < 16; r++) red[wave][(t * 16 + r) * 64 + lane] = acc[t][r];
  __syncthreads();
  // epilogue: the W*64 threads share the TM*1024 outputs; element (t, r, lane') sits at
  // row 32t + 8(r/4) + 4(lane'/32) + r%4, column lane'%32
  for (int e = tid; e < TM * 1024; e += W * 64) {
    const int l2 = e & 63, r = (e >> 6) & 15, t = e >> 10;
    const int row = m0 + 32 * t + 8 * (r / 4) + 4 * (l2 >> 5) + (r % 4), col = n0 + (l2 & 31);
    if (row >= g.M || col >= g.N) continue;
    float s = red[0][e];
#pragma unroll
    for (int w = 1; w < W; w++) s += red[w][e];
    float v = padding_column(g, col) ? 0.f : g.alpha * s;
    if (g.beta != 0.f) v += g.beta * g.C[row * g.ldc + col];
    if (g.D) v += g.D[(long)(row >> g.dshift) * g.ldd + col];
    g.C[row * g.ldc + col] = v;
  }
}

struct GemmPlan {
  enum Kind { TILE128, TILE64, SKINNY } kind;
  int splits;   // > 1: partial tiles to the workspace + reduce kernel (TILE64 only)
  int kchunk;
  long tiles;
};

static bool skinny_ok(int tA, int tB, int K, const float *A, int lda, const float *B, int ldb) {
  if (tA || K % 4 || lda % 4 || !aligned16(A)) return false;
  if (tB && (ldb % 4 || !aligned16(B))) return false;
  return true;
}

// Rows of a k-contiguous operand further apart than the large tile's 32-bit offsets reach.
static bool far_rows(int tA, int tB, int lda, int ldb) { return (!tA && lda >= 1 << 23) || (tB && ldb >= 1 << 23); }

static GemmPlan plan_gemm(int tA, int tB, int M, int N, int K, bool skinny_allowed, bool allow_split, bool large_ok = true) {
  GemmPlan p;
  const long cus = num_cus();
  const long t128 = (long)((M + 127) / 128) * ((N + 127) / 128);
  const long t64 = (long)((M + 63) / 64) * ((N + 63) / 64);
  auto split = [&](GemmPlan::Kind kind, long tiles, long s) {
    p.kind = kind;
    p.tiles = tiles;
    p.kchunk = K;
    p.splits = 1;
    if (s > 1) {
      p.kchunk = (int)(((K + s - 1) / s + 31) / 32 * 32);
      p.splits = (K + p.kchunk - 1) / p.kchunk;
    }
    return p;
  };
  // A CU holds two or three workgroups of the large tile; from two per CU on it is the faster one (4700 x 2048 x
  // 300, 592 tiles: 44.6 us against 49.8; 2368 rows, 304 tiles: 31.1 against 27.3).
  if (large_ok && t128 >= 2 * cus) return split(GemmPlan::TILE128, t128, 1);
  // Fewer large tiles: K is split until about three share a CU, if that leaves each split at least 512 of K
  // (4000 x 1024 x 3072: 150 us against 170 on the small tile).  (A CU holds two of them beyond 512 of K,
  // gemm_split.h.  Splits for two are 1 to 6 % faster -- TN 1024 x 4096 x 73000 3421 us against 3462, 512 x 2048 x
  // 7088 94 against 98.5 -- but the size of the partials decides what cavs_sgemm_splitk_static refuses.)
  if (large_ok && allow_split && 4 * t128 >= cus && K >= 2048) {
    long s = (3 * cus + t128 - 1) / t128;
    // one or two more splits when they even out the workgroups per CU; ties keep the fewer splits
    // (less partial traffic)
    auto fill = [&](long sp) {
      const long w = t128 * sp, rounds = (w + cus - 1) / cus;
      return (double)w / (double)(rounds * cus);
    };
    for (long c = s + 1; c <= s + 2; c++)
      if (fill(c) > fill(s) + 0.02) s = c;
    s = std::min<long>(s, K / 512);
    if (t128 * s >= 2 * cus) return split(GemmPlan::TILE128, t128, s);
  }
  if (t64 >= 2 * cus || K < 64) return split(GemmPlan::TILE64, t64, 1);
  // the skinny kernel reads a k-contiguous B (NT) sixteen bytes per lane and row, which only
  // pays for a handful of rows; with B row-major (NN) it holds up to about a thousand
  if (skinny_allowed && M <= (tB ? 128 : 1024)) {
    p.kind = GemmPlan::SKINNY;
    p.splits = 1;
    p.kchunk = K;
    p.tiles = t64;
    return p;
  }
  long s = 1;
  if (allow_split && K >= 256) {
    s = std::min({(3 * cus + t64 - 1) / t64, (long)(K / 128), 32L});  // at least 128 of K per split
  }
  return split(GemmPlan::TILE64, t64, s);
}

// The plan of a product of which `expect` rows of C (or of K) are thought to take part: tiles for all of them.
static GemmPlan plan_live(int tA, int tB, int M, int N, int K, int lda, int ldb, bool allow_split, int expect) {
  const int m = tA ? M : std::min(M, std::max(expect, 1)), k = tA ? std::min(K, std::max(expect, 1)) : K;
  GemmPlan p = plan_gemm(tA, tB, m, N, k, false, allow_split, !far_rows(tA, tB, lda, ldb));
  const int tile = p.kind == GemmPlan::TILE128 ? 128 : 64;
  p.tiles = (long)((M + tile - 1) / tile) * ((N + tile - 1) / tile);
  if (tA) p.kchunk = K;  // (set by the kernel)
  return p;
}

static GemmPlan plan_product(const cavs_gemm_desc &q) {
  return q.live ? plan_live(q.transA, q.transB, q.M, q.N, q.K, q.lda, q.ldb, true, q.live_expect)
                : plan_gemm(q.transA, q.transB, q.M, q.N, q.K, false, true, !far_rows(q.transA, q.transB, q.lda, q.ldb));
}

static size_t plan_workspace(const GemmPlan &p, int M, int N) {
  return p.splits > 1 ? sizeof(float) * (size_t)p.splits * M * N : 0;
}

static bool vec_path_ok(const GemmArgs &g, int tA, int tB) {
  if (!aligned16(g.A) || !aligned16(g.B) || g.lda % 4 || g.ldb % 4) return false;
  // the contiguous index of each operand must come in whole float4s
  if (!tA ? (g.K % 4) : (g.M % 4)) return false;
  if (tB ? (g.K % 4) : (g.N % 4)) return false;
  return true;
}

// LDS a tile launch of the calling thread asks for on top of its panels (cavs_sgemm_group_beside): the
// workgroups then take more of a CU than they use, and fewer of them share one
static thread_local unsigned t_lds_pad = 0;

// The grid of a launch of BM x BN tiles: a known block of whole row tiles becomes a launch of its own (GemmArgs::seg_rows).
static dim3 tile_grid(GemmArgs *g, int BM, int BN, const GemmPlan &p) {
  dim3 grid((unsigned)p.tiles, p.splits);
  if (g->live) {  // (the kernel counts its tiles; room for two padded launches)
    grid.x = (unsigned)((p.tiles + 7) / 8 * 8 + 8);
    return grid;
  }
  if (g->zkind == CAVS_GEMM_A_ZERO || g->zkind == CAVS_GEMM_C_UNUSED) {
    const int tilesM = (g->M + BM - 1) / BM, tilesN = (g->N + BN - 1) / BN, rows = std::min(g->zrows, g->M);
    if (rows / BM > 0 && rows / BM < tilesM) {
      const bool unused = g->zkind == CAVS_GEMM_C_UNUSED;
      g->seg_rows = rows / BM;
      g->seg_cols = unused ? std::min((g->zcol + BN - 1) / BN, tilesN) : tilesN;
      g->seg_mixed = unused ? (rows + BM - 1) / BM : g->seg_rows;
      auto whole = [](long n) { return (n + 7) / 8 * 8; };
      grid.x = (unsigned)(whole((long)g->seg_rows * g->seg_cols) + whole((long)(g->seg_mixed - g->seg_rows) * tilesN) +
                          whole((long)(tilesM - g->seg_mixed) * tilesN) + whole((long)g->seg_rows * (tilesN - g->seg_cols)));
    }
  }
  return grid;
}

template <int BM, int BN, int BK, bool FOLD>
static void launch_split(const GemmArgs &args, int tA, int tB, bool vec, const GemmPlan &p, hipStream_t st) {
  GemmArgs g = args;
  const dim3 grid = tile_grid(&g, BM, BN, p), block(kThreads);
#define CAVS_GEMM_CASE(TA, TB)                                                                                \
  if (vec)                                                                                                    \
    launch(sgemm_split_kernel<BM, BN, BK, TA, TB, true, FOLD>, grid, block, t_lds_pad, st, g);                \
  else                                                                                                        \
    launch(sgemm_split_kernel<BM, BN, BK, TA, TB, false, FOLD>, grid, block, t_lds_pad, st, g)
  if (!tA && !tB) { CAVS_GEMM_CASE(false, false); }
  else if (!tA && tB) { CAVS_GEMM_CASE(false, true); }
  else if (tA && !tB) { CAVS_GEMM_CASE(true, false); }
  else { CAVS_GEMM_CASE(true, true); }
#undef CAVS_GEMM_CASE
}

static int check_gemm(const char *who, int tA, int tB, int M, int N, int K, const float *A, int lda,
                      const float *B, int ldb, const float *C, int ldc) {
  CAVS_REQUIRE(M >= 0 && N >= 0 && K >= 0, "%s: negative dimension M=%d N=%d K=%d", who, M, N, K);
  if (M == 0 || N == 0) return CAVS_OK;
  CAVS_REQUIRE(C && ldc >= N, "%s: bad C (ldc=%d, N=%d)", who, ldc, N);
  if (K > 0) {
    CAVS_REQUIRE(A && B, "%s: null operand", who);
    CAVS_REQUIRE(lda >= (tA ? M : K), "%s: lda=%d too small", who, lda);
    CAVS_REQUIRE(ldb >= (tB ? K : N), "%s: ldb=%d too small", who, ldb);
  }
  return CAVS_OK;
}

template <bool TB>
static void launch_skinny(const GemmArgs &g, hipStream_t st) {
  constexpr int W = 8;
  if (g.M <= 32) {
    dim3 grid((g.N + 31) / 32, 1);
    launch(sgemm_skinny_kernel<1, TB, W>, grid, W * 64, 0, st, g);
  } else {
    dim3 grid((g.N + 31) / 32, (g.M + 63) / 64);
    launch(sgemm_skinny_kernel<2, TB, W>, grid, W * 64, 0, st, g);
  }
}

// the looked-up rows of cavs_embed_pull_sgemm (GemmArgs::pull_*)
struct PullRows {
  const int *rows;
  const float *x;
  float *copy;
  long ld_copy;
  float *ids;
};

// What the caller knows about a block of an operand or of the result (cavs_gemm_desc::zero_kind,
// zero_rows, zero_col).  It is a licence, not an order: set() keeps it only in the forms the tile
// routine acts on and the kernels that never look at it give the plain product.
struct BlockHint {
  int kind = 0, rows = 0, col = 0;
  void set(GemmArgs *g, int tA, int tB, bool plain_store) const {
    if (rows <= 0 || col < 0) return;
    const bool ok = (kind == CAVS_GEMM_C_UNUSED && plain_store && col > 0) || (kind == CAVS_GEMM_A_ZERO && !tA && col % 4 == 0) ||
                    (kind == CAVS_GEMM_B_ZERO && !tB);
    if (!ok) return;
    g->zkind = kind;
    g->zrows = rows;
    g->zcol = col;
  }
};

// cavs_gemm_desc::pad_block, pad_used
struct Padding {
  int block = 0, used = 0;
};

static int run_gemm(const char *who, int tA, int tB, int M, int N, int K, float alpha, const float *A,
                    int lda, const float *B, int ldb, float beta, float *C, int ldc, const float *D,
                    int ldd, int dshift, void *ws, size_t ws_bytes, void *stream, const PullRows *pull = nullptr,
                    const BlockHint *hint = nullptr, const int *live = nullptr, int live_expect = 0, Padding pad = {},
                    const float *row_ids = nullptr) {
  int rc = check_gemm(who, tA, tB, M, N, K, A, lda, B, ldb, C, ldc);
  if (rc || M == 0 || N == 0) return rc;
  // Looked-up rows: up to 128 of them the skinny kernel, beyond it the 64 x 64 tiles (M x 2048 x 300..512: 21
  // rows 12.4 -> 7.9 us, 120 rows 19.7 -> 15.1, 300 rows 20.5 and 26.2).
  GemmPlan p = live ? plan_live(tA, tB, M, N, K, lda, ldb, ws != nullptr, live_expect)
                    : plan_gemm(tA, tB, M, N, K, (!pull || M <= 128) && skinny_ok(tA, tB, K, A, lda, B, ldb), ws != nullptr,
                                !pull && !far_rows(tA, tB, lda, ldb));
  hipStream_t st = as_stream(stream);
  GemmArgs g{M, N, K, A, lda, B, ldb, C, ldc, alpha, beta, D, ldd, dshift, p.kchunk, nullptr};
  g.live = live;
  g.pad_block = pad.block;
  g.pad_used = pad.used;
  g.row_ids = row_ids;
  if (hint) hint->set(&g, tA, tB, beta == 0.f && !D);
  if (pull) {
    g.pull_rows = pull->rows;
    g.pull_x = pull->x;
    g.pull_copy = pull->copy;
    g.ld_copy = pull->ld_copy;
    g.pull_ids = pull->ids;
  }
  if (p.kind == GemmPlan::SKINNY) {
    if (tB) launch_skinny<true>(g, st); else launch_skinny<false>(g, st);
    CAVS_LAUNCH_CHECK();
    return CAVS_OK;
  }
  if (p.splits > 1) {
    size_t need = plan_workspace(p, M, N);
    CAVS_REQUIRE(ws_bytes >= need && aligned16(ws), "%s: workspace of %zu bytes needed, %zu given", who, need, ws_bytes);
    g.ws = static_cast<float *>(ws);
  }
  bool vec = vec_path_ok(g, tA, tB);
  if (pull) {
    const dim3 grid = tile_grid(&g, 64, 64, p), block(kThreads);
    if (vec) launch(sgemm_split_kernel<64, 64, 16, false, false, true, true, true>, grid, block, 0, st, g);
    else launch(sgemm_split_kernel<64, 64, 16, false, false, false, true, true>, grid, block, 0, st, g);
  } else if (p.kind == GemmPlan::TILE128) {
    if (K > 2 * kSplitChain) launch_split<128, 128, 16, true>(g, tA, tB, vec, p, st);
    else launch_split<128, 128, 16, false>(g, tA, tB, vec, p, st);
  } else {
    launch_split<64, 64, 16, true>(g, tA, tB, vec, p, st);
  }
  CAVS_LAUNCH_CHECK();
  if (p.splits > 1) {
    long total = (long)M * N;
    launch(splitk_reduce_kernel, (unsigned)((total + 255) / 256), 256, 0, st, g, p.splits, tA != 0);
    CAVS_LAUNCH_CHECK();
  }
  return CAVS_OK;
}

// Plans a group: every product on the 64x64 tile, K split so that all workgroups of the group
// together are about four per CU (what a CU holds at once; inside a training step eight per CU
// measured no better, though it is in a back-to-back loop), each with at least 256 of K; 128 where the workgroups
// are few even so, and a single product is cut as it would be by itself (plan_product).
// `tail_product` >= 0: that product's result is handed on to the embedding scatter-add (dtable, ids)
// and `counters` [n_counters]: the group's launch adds up its splits itself where they are enough (GroupFold)
struct Lookups {  // bit p: product p is over the rows that the ids looked up, equal where those are (GemmArgs::row_ids)
  unsigned products = 0;
  int from = 0;
};
static int run_group(int count, const cavs_gemm_desc *d, void *ws, size_t ws_bytes, size_t *need_out, void *stream,
                     int tail_product = -1, float *dtable = nullptr, const float *ids = nullptr, int *counters = nullptr, int n_counters = 0, const cavs_colsum_desc *sums = nullptr, Lookups lookups = {}) {
  CAVS_REQUIRE(count >= 0 && count <= kGroupMax, "cavs_sgemm_group: %d products, at most %d", count, kGroupMax);
  CAVS_REQUIRE(count == 0 || d, "cavs_sgemm_group: null descriptors");
  EmbedTail tail{};
  if (tail_product >= 0 && !need_out) {
    CAVS_REQUIRE(tail_product < count, "cavs_sgemm_group_embed_bwd: product %d of %d", tail_product, count);
    const cavs_gemm_desc &q = d[tail_product];
    CAVS_REQUIRE(q.alpha == 1.f && q.beta == 0.f, "cavs_sgemm_group_embed_bwd: the product that feeds the table takes alpha = 1, beta = 0");
    CAVS_REQUIRE((q.M == 0 || q.N == 0) || (dtable && ids), "cavs_sgemm_group_embed_bwd: null pointer");
    // unsplit (or run alone): the scatter-add reads C
    tail = EmbedTail{dtable, ids, q.C, q.ldc, 0, 1, nullptr, 0, q.M, q.N, (q.M + kEmbedRows - 1) / kEmbedRows,
                     q.live};
  }
  GemmGroup G{}, R{};
  GroupFold F{};
  F.embed = -1;
  long split_tiles = 0;
  auto looked_up = [&](int p) {
    const cavs_gemm_desc &q = d[p];
    return (lookups.products >> p & 1) && !q.live && (q.transA ? !q.transB : q.transB && p == tail_product);
  };
  // K as the plan sees it, and the number of tiles it expects (cavs_gemm_desc::live)
  auto plan_K = [](const cavs_gemm_desc &q) { return q.live && q.transA ? std::min(q.K, std::max(q.live_expect, 1)) : q.K; };
  auto plan_tiles = [](const cavs_gemm_desc &q) {
    const int m = q.live && !q.transA ? std::min(q.M, std::max(q.live_expect, 1)) : q.M;
    return (long)((m + 63) / 64) * ((q.N + 63) / 64);
  };
  double work = 0;
  long tiles[kGroupMax];
  bool alone[kGroupMax];
  int grouped = 0;
  size_t most = 0;
  for (int p = 0; p < count; p++) {
    const cavs_gemm_desc &q = d[p];
    if (!need_out) {
      int rc = check_gemm("cavs_sgemm_group", q.transA, q.transB, q.M, q.N, q.K, q.A, q.lda, q.B, q.ldb, q.C, q.ldc);
      if (rc) return rc;
    }
    CAVS_REQUIRE(q.M >= 0 && q.N >= 0 && q.K >= 0, "cavs_sgemm_group: negative dimension in product %d", p);
    CAVS_REQUIRE(q.pad_block >= 0 && q.pad_used >= 0, "cavs_sgemm_group: bad padding in product %d (block %d, used %d)", p, q.pad_block, q.pad_used);
    CAVS_REQUIRE(q.zero_kind >= 0 && q.zero_kind <= CAVS_GEMM_B_ZERO && q.zero_rows >= 0 && q.zero_col >= 0,
                 "cavs_sgemm_group: bad block hint in product %d (kind %d, rows %d, col %d)", p, q.zero_kind, q.zero_rows, q.zero_col);
    tiles[p] = (long)((q.M + 63) / 64) * ((q.N + 63) / 64);
    // a product that fills the chip with large tiles by itself is better off on them, alone
    alone[p] = q.M > 0 && q.N > 0 && plan_product(q).kind == GemmPlan::TILE128;
    if (!alone[p] && q.M > 0 && q.N > 0) grouped++;
  }
  for (int p = 0; p < count; p++) {
    const cavs_gemm_desc &q = d[p];
    if (q.M == 0 || q.N == 0) continue;
    if (!alone[p] && (grouped >= 2 || counters || need_out)) {
      work += (double)plan_tiles(q) * plan_K(q);
      if (grouped < 2 && need_out) most = std::max(most, plan_workspace(plan_product(q), q.M, q.N));  // (for either way)
      continue;
    }
    alone[p] = true;
    most = std::max(most, plan_workspace(plan_product(q), q.M, q.N));
  }
  const long slots = 4 * num_cus();
  long kc = (long)(work / (double)slots);
  kc = (kc + 31) / 32 * 32;
  if (kc < 256) kc = 256;
  // The chip holds `slots` of these workgroups at once.  A launch of a few more runs them as a
  // second round behind the first -- a whole workgroup's time for a handful of tiles (measured:
  // 1024 workgroups 95 us, 1032 workgroups 122 us) -- so the k chunk grows until the launch fits,
  // unless the tiles alone overflow it.
  auto launch_size = [&](long chunk) {
    long total = 0;
    for (int p = 0; p < count; p++) {
      const cavs_gemm_desc &q = d[p];
      if (q.M == 0 || q.N == 0 || alone[p]) continue;
      const long K = plan_K(q);
      long s = K > 0 ? (K + chunk / 2) / chunk : 1;
      if (s < 1) s = 1;
      const long kchunk = K > 0 ? ((K + s - 1) / s + 31) / 32 * 32 : 1;
      const long splits = K > 0 ? (K + kchunk - 1) / kchunk : 1;
      total += (plan_tiles(q) * splits + 7) / 8 * 8;
    }
    return total;
  };
  if (launch_size(1L << 30) <= slots)
    while (launch_size(kc) > slots) kc += 32;
  // Few workgroups: a step of K is a latency then, not work (the head of 840 vertices, H = 224, 23 classes, 72 workgroups: 14.7 us in
  // chunks of 256, 12.4 in chunks of 128)
  while (kc > 128 && launch_size(kc / 2) <= 2 * num_cus()) kc /= 2;
  size_t need = 0;
  bool vec = true;
  int n = 0, nr = 0;
  for (int p = 0; p < count; p++) {
    const cavs_gemm_desc &q = d[p];
    if (q.M == 0 || q.N == 0 || alone[p]) continue;
    const int K = plan_K(q);
    long s = K > 0 ? (K + kc / 2) / kc : 1;
    if (s < 1) s = 1;
    int kchunk = K > 0 ? (int)(((K + s - 1) / s + 31) / 32 * 32) : 1;
    int splits = K > 0 ? (K + kchunk - 1) / kchunk : 1;
    if (grouped == 1) {  // as it would be cut by itself
      const GemmPlan alone_plan = plan_product(q);
      kchunk = alone_plan.kchunk;
      splits = alone_plan.splits;
    }
    GemmArgs g{q.M, q.N, q.K, q.A, q.lda, q.B, q.ldb, q.C, q.ldc, q.alpha, q.beta, nullptr, 0, 0, kchunk, nullptr};
    g.live = q.live;
    g.pad_block = q.pad_block;
    g.pad_used = q.pad_used;
    BlockHint{q.zero_kind, q.live ? 1 : q.zero_rows, q.zero_col}.set(&g, q.transA, q.transB, q.beta == 0.f);
    G.long_tiles[n] = (int)tiles[p];
    G.long_splits[n] = splits;
    if (looked_up(p)) {
      g.row_ids = ids;
      g.ids_from = lookups.from;
      const long rows = std::min<long>(((long)lookups.from + 63) / 64 * ((q.N + 63) / 64), tiles[p]);
      if (q.transA) G.long_splits[n] = (int)std::min<long>(((long)lookups.from + kchunk - 1) / kchunk, splits);
      else G.long_tiles[n] = (int)rows;
    }
    if (splits > 1) {
      if (ws) g.ws = reinterpret_cast<float *>(static_cast<char *>(ws) + need);
      need += ((size_t)splits * q.M * q.N * sizeof(float) + 255) / 256 * 256;
    }
    if (!need_out && !vec_path_ok(g, q.transA, q.transB)) vec = false;
    G.g[n] = g;
    G.tiles[n] = (int)tiles[p];
    G.splits[n] = splits;
    G.form[n] = (q.transA ? 2 : 0) + (q.transB ? 1 : 0);
    const long first = (long)G.long_tiles[n] * G.long_splits[n];
    G.first[n + 1] = G.first[n] + (int)((first + 7) / 8 * 8);
    G.after[n + 1] = G.after[n] + (int)((tiles[p] * splits - first + 7) / 8 * 8);
    if (splits > 1) {
      F.first[n] = (int)split_tiles;
      split_tiles += tiles[p];
    }
    if (p == tail_product) F.embed = n;
    n++;
    if (splits > 1 && p == tail_product && !need_out) {
      // the scatter-add sums this product's partials itself (and leaves the sum in C as well)
      tail.dy = g.ws;
      tail.ld_dy = q.N;
      tail.part_stride = (long)q.M * q.N;
      tail.parts = splits;
      tail.copy = q.C;
      tail.ld_copy = q.ldc;
    } else if (splits > 1) {
      R.g[nr] = g;
      R.splits[nr] = splits;
      R.form[nr] = q.transA ? 2 : 0;
      R.first[nr + 1] = R.first[nr] + (int)(((long)q.M * q.N + 255) / 256);
      nr++;
    }
  }
  G.count = n;
  R.count = nr;
  need = std::max(need, most);
  if (need_out) {
    *need_out = need;
    return CAVS_OK;
  }
  CAVS_REQUIRE(need == 0 || (ws && ws_bytes >= need && aligned16(ws)), "cavs_sgemm_group: workspace of %zu bytes needed, %zu given", need, ws_bytes);
  // the products that run alone share the workspace with the group: the stream orders them
  for (int p = 0; p < count; p++) {
    const cavs_gemm_desc &q = d[p];
    if (q.M == 0 || q.N == 0 || !alone[p]) continue;
    const BlockHint hint{q.zero_kind, q.live ? 1 : q.zero_rows, q.zero_col};
    int rc = run_gemm("cavs_sgemm_group", q.transA, q.transB, q.M, q.N, q.K, q.alpha, q.A, q.lda, q.B, q.ldb, q.beta,
                      q.C, q.ldc, nullptr, 0, 0, ws, ws_bytes, stream, nullptr, &hint, q.live, q.live_expect, {q.pad_block, q.pad_used});
    if (rc) return rc;
  }
  hipStream_t st = as_stream(stream);
  bool with_tail = tail_product >= 0 && tail.n > 0 && tail.E > 0;
  if (counters && n > 0 && split_tiles <= n_counters) {
    F.counters = counters;
    F.tail = tail;
    if (!with_tail) F.embed = -1;
    if (F.embed >= 0) with_tail = false;
    nr = R.count = 0;
  }
  unsigned grid = G.first[n] + G.after[n];
  if (sums && sums->n > 0 && n > 0) {
    F.sums = colsum_job(sums->parts, sums->inp, sums->ld, sums->n, sums->w);
    grid += (unsigned)((sums->w + 63) / 64 * F.sums.chunks);
  } else if (sums) {
    int rc = cavs_colsum_blocks(nullptr, sums->inp, sums->ld, sums->n, sums->w, 1, nullptr, sums->parts,
                                cavs_colsum_blocks_workspace(sums->n, sums->w, 1), stream);
    if (rc) return rc;
  }
  if (n > 0) {
    if (vec) launch(sgemm_group_kernel<true>, grid, kThreads, 0, st, G, F);
    else launch(sgemm_group_kernel<false>, grid, kThreads, 0, st, G, F);
    CAVS_LAUNCH_CHECK();
  }
  if (with_tail) {
    const int gy = (tail.E + kEmbedCols - 1) / kEmbedCols;
    launch(splitk_reduce_group_embed_kernel, (unsigned)(R.first[nr] + tail.gx * gy), 256, 0, st, R, tail);
    CAVS_LAUNCH_CHECK();
  } else if (nr > 0) {
    launch(splitk_reduce_group_kernel, (unsigned)R.first[nr], 256, 0, st, R);
    CAVS_LAUNCH_CHECK();
  }
  return CAVS_OK;
}

// Split-K partials of cavs_sgemm_splitk_static: device memory that exists from the moment the
// code object is loaded, so that entry point never has to ask the allocator for any.  Every GPU
// the library runs on holds its own copy until the process ends.
constexpr size_t kStaticScratchBytes = size_t(32) << 20;
constexpr int kStaticScratchDevices = 64;
static __device__ __align__(256) float scratch[kStaticScratchBytes / sizeof(float)];
// Device address of `scratch` on each GPU (the array's name is only a host-side stand-in for the
// symbol; kernels, fills and copies take the address looked up here).
static std::atomic<float *> g_scratch_ptr[kStaticScratchDevices];

// Looks the address up for the current device, once (two threads that both find it missing look
// it up twice and store the same value).
int static_scratch_setup(float **out) {
  int dev = 0;
  CAVS_HIP_TRY(hipGetDevice(&dev));
  CAVS_REQUIRE(dev >= 0 && dev < kStaticScratchDevices, "static scratch: device %d out of range", dev);
  float *ptr = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (!ptr) {
    CAVS_HIP_TRY(hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(scratch)));
    CAVS_REQUIRE(ptr && aligned16(ptr), "static scratch: no usable address on device %d", dev);
    g_scratch_ptr[dev].store(ptr, std::memory_order_release);
  }
  if (out) *out = ptr;
  return CAVS_OK;
}

}  // namespace cavs

using namespace cavs;

extern "C" {

int cavs_mfma_probe(float *out, size_t out_floats, int iters, double *flops, void *stream) {
  const int blocks = 4 * num_cus();
  CAVS_REQUIRE(out && iters > 0 && out_floats >= (size_t)blocks * 256, "cavs_mfma_probe: output of %d floats needed", blocks * 256);
  launch(mfma_probe_kernel, blocks, 256, 0, as_stream(stream), out, iters);
  CAVS_LAUNCH_CHECK();
  if (flops) *flops = (double)blocks * 4 * iters * 8 * 2.0 * 32 * 32 * 2;
  return CAVS_OK;
}

size_t cavs_sgemm_splitk_static_max_bytes(void) { return kStaticScratchBytes; }

int cavs_sgemm_splitk_static(int transA, int transB, int M, int N, int K, float alpha, const float *A,
                             int lda, const float *B, int ldb, float beta, float *C, int ldc, void *stream) {
  float *ptr = nullptr;
  int rc = static_scratch_setup(&ptr);
  if (rc) return rc;
  if (M > 0 && N > 0 && K > 0) {
    // the same plan run_gemm makes when it is handed a workspace
    GemmPlan p = plan_gemm(transA, transB, M, N, K, skinny_ok(transA, transB, K, A, lda, B, ldb), true);
    size_t need = p.kind == GemmPlan::SKINNY ? 0 : plan_workspace(p, M, N);
    if (need > kStaticScratchBytes)
      return set_error(CAVS_EINVAL,
                       "cavs_sgemm_splitk_static: M=%d N=%d K=%d needs %zu bytes of split-K partials, the built-in "
                       "scratch holds %zu; use cavs_sgemm_splitk with a workspace of the caller's",
                       M, N, K, need, kStaticScratchBytes);
  }
  // partials are written before they are read, every element of them: nothing of the previous
  // call's contents has to be cleared
  return run_gemm("cavs_sgemm_splitk_static", transA, transB, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc,
                  nullptr, 0, 0, ptr, kStaticScratchBytes, stream);
}

size_t cavs_sgemm_group_workspace(int count, const cavs_gemm_desc *products) {
  size_t need = 0;
  if (run_group(count, products, nullptr, 0, &need, nullptr) != CAVS_OK) return 0;
  return need;
}

int cavs_sgemm_group(int count, const cavs_gemm_desc *products, void *workspace, size_t workspace_bytes,
                     void *stream) {
  return run_group(count, products, workspace, workspace_bytes, nullptr, stream);
}

int cavs_sgemm_group_once(int count, const cavs_gemm_desc *products, int embed_product, float *dtable, const float *ids, void *workspace,
                          size_t workspace_bytes, int *counters, int n_counters, const cavs_colsum_desc *sums, void *stream) {
  CAVS_REQUIRE(counters && n_counters >= 0, "cavs_sgemm_group_once: null counters");
  CAVS_REQUIRE(!sums || (sums->n >= 0 && sums->w > 0 && sums->ld >= sums->w && sums->parts && (sums->inp || sums->n == 0)),
               "cavs_sgemm_group_once: bad column sums");
  return run_group(count, products, workspace, workspace_bytes, nullptr, stream, embed_product, dtable, ids, counters, n_counters, sums);
}

int cavs_sgemm_group_lookups(int count, const cavs_gemm_desc *products, int embed_product, float *dtable, const float *ids, unsigned lookup_products,
                             int same_from, void *workspace, size_t workspace_bytes, int *counters, int n_counters, const cavs_colsum_desc *sums,
                             void *stream) {
  CAVS_REQUIRE(counters && n_counters >= 0, "cavs_sgemm_group_lookups: null counters");
  CAVS_REQUIRE(embed_product >= 0 && same_from >= 0, "cavs_sgemm_group_lookups: product %d, rows from %d", embed_product, same_from);
  CAVS_REQUIRE(!sums || (sums->n >= 0 && sums->w > 0 && sums->ld >= sums->w && sums->parts && (sums->inp || sums->n == 0)),
               "cavs_sgemm_group_lookups: bad column sums");
  return run_group(count, products, workspace, workspace_bytes, nullptr, stream, embed_product, dtable, ids, counters, n_counters, sums,
                   {lookup_products, same_from});
}

int cavs_sgemm_group_beside(int count, const cavs_gemm_desc *products, void *workspace, size_t workspace_bytes,
                            void *stream) {
  // With the 48 KB of a large tile's panels more than half of a CU's LDS: one workgroup to a CU.  (Two of them, at
  // 232 registers, leave no room for the chain's wavefronts.  Training steps of chain LSTMs with a head of 10000
  // at H = 640, 768, 1024: 2.97, 4.70, 6.03 ms against 3.16, 5.00, 6.20.)
  t_lds_pad = 34u << 10;
  const int rc = run_group(count, products, workspace, workspace_bytes, nullptr, stream);
  t_lds_pad = 0;
  return rc;
}

int cavs_sgemm_group_embed_bwd(int count, const cavs_gemm_desc *products, int embed_product, float *dtable, const float *ids,
                               void *workspace, size_t workspace_bytes, void *stream) {
  CAVS_REQUIRE(embed_product >= 0, "cavs_sgemm_group_embed_bwd: product %d", embed_product);
  return run_group(count, products, workspace, workspace_bytes, nullptr, stream, embed_product, dtable, ids);
}

int cavs_embed_pull_sgemm(float *C, int ldc, float *e_out, int ld_e, float *ids_out, const float *x, const int *rows,
                          const float *table, int n, int E, const float *B, int ldb, int N, int unused_rows, int unused_col,
                          void *stream) {
  return cavs_embed_pull_sgemm_padded(C, ldc, e_out, ld_e, ids_out, x, rows, table, n, E, B, ldb, N, unused_rows, unused_col, 0, 0, stream);
}

int cavs_embed_pull_sgemm_padded(float *C, int ldc, float *e_out, int ld_e, float *ids_out, const float *x, const int *rows,
                                 const float *table, int n, int E, const float *B, int ldb, int N, int unused_rows, int unused_col,
                                 int pad_block, int pad_used, void *stream) {
  CAVS_REQUIRE(n >= 0 && E > 0 && N >= 0 && ld_e >= E, "cavs_embed_pull_sgemm: bad shape n=%d E=%d N=%d ld_e=%d", n, E, N, ld_e);
  CAVS_REQUIRE(pad_block >= 0 && pad_used >= 0, "cavs_embed_pull_sgemm: bad padding (block %d, used %d)", pad_block, pad_used);
  CAVS_REQUIRE(unused_rows >= 0 && unused_col >= 0, "cavs_embed_pull_sgemm: bad unused block (rows %d, col %d)", unused_rows, unused_col);
  const BlockHint hint{CAVS_GEMM_C_UNUSED, unused_rows, unused_col};
  if (n == 0) return CAVS_OK;
  CAVS_REQUIRE(e_out && ids_out && x && rows && table, "cavs_embed_pull_sgemm: null pointer");
  // the copy goes out in whole float4s on the vector path
  CAVS_REQUIRE(E % 4 != 0 || (aligned16(e_out) && ld_e % 4 == 0), "cavs_embed_pull_sgemm: e_out must be 16-byte aligned with ld_e a multiple of 4");
  // A product large enough for the 128 x 128 tiles gains nothing from the saved launch and its
  // workgroups are slowed by the lookups (7331 x 2048 x 512: 157 -> 180 us): the two calls then.
  if (N == 0 || plan_gemm(0, 0, n, N, E, false, false).kind == GemmPlan::TILE128) {
    int rc = cavs_embed_pull_fwd(e_out, ld_e, ids_out, x, rows, table, n, E, stream);
    if (rc || N == 0) return rc;
    return run_gemm("cavs_embed_pull_sgemm", 0, 0, n, N, E, 1.f, e_out, ld_e, B, ldb, 0.f, C, ldc, nullptr, 0, 0, nullptr, 0, stream,
                    nullptr, &hint, nullptr, 0, {pad_block, pad_used}, ids_out);
  }
  const PullRows pull{rows, x, e_out, ld_e, ids_out};
  return run_gemm("cavs_embed_pull_sgemm", 0, 0, n, N, E, 1.f, table, E, B, ldb, 0.f, C, ldc, nullptr, 0, 0, nullptr, 0, stream, &pull,
                  &hint, nullptr, 0, {pad_block, pad_used});
}

int cavs_sgemm(int transA, int transB, int M, int N, int K, float alpha, const float *A, int lda,
               const float *B, int ldb, float beta, float *C, int ldc, void *stream) {
  return run_gemm("cavs_sgemm", transA, transB, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, nullptr, 0,
                  0, nullptr, 0, stream);
}

int cavs_sgemm_addrows(int transA, int transB, int M, int N, int K, const float *A, int lda,
                       const float *B, int ldb, const float *D, int ldd, int d_shift, float *C,
                       int ldc, void *workspace, size_t workspace_bytes, void *stream) {
  if (M > 0 && N > 0)
    CAVS_REQUIRE(D && ldd >= N && d_shift >= 0 && d_shift < 31, "cavs_sgemm_addrows: bad addend (ldd=%d shift=%d)", ldd, d_shift);
  return run_gemm("cavs_sgemm_addrows", transA, transB, M, N, K, 1.f, A, lda, B, ldb, 0.f, C, ldc, D, ldd,
                  d_shift, workspace, workspace_bytes, stream);
}

size_t cavs_sgemm_splitk_workspace(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  // sized for the split plan whether or not a given call ends up taking the skinny path
  return std::max(plan_workspace(plan_gemm(0, 0, M, N, K, false, true), M, N), plan_workspace(plan_gemm(0, 0, M, N, K, false, true, false), M, N));
}

int cavs_sgemm_splitk(int transA, int transB, int M, int N, int K, float alpha, const float *A,
                      int lda, const float *B, int ldb, float beta, float *C, int ldc,
                      void *workspace, size_t workspace_bytes, void *stream) {
  return run_gemm("cavs_sgemm_splitk", transA, transB, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc,
                  nullptr, 0, 0, workspace, workspace_bytes, stream);
}

}  // extern "C"
