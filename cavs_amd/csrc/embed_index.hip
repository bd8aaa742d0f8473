// The words of a batch, each once: a table row that many vertices look up (every internal vertex of a
// parse tree looks up row 0, text repeats its frequent words) is multiplied by W once, the gradients
// of the vertices that read it are added up first, and the products of the backward pass run over words
// instead of vertices.
//   cavs_embed_index   sorts the vertices by id: up to three sweeps of a radix sort with stable ranks,
//                      then the segments of equal ids; in one workgroup while it all fits LDS
//   cavs_embed_words   the table rows of the words
//   cavs_spread_rows   a word's row of x * W to every vertex that looked it up
//   cavs_gather_sums   a word's gradient row: the sum over its vertices, in vertex order
#include <algorithm>

#include "common.h"

namespace cavs {

constexpr int kIndexThreads = 1024, kIndexWaves = kIndexThreads / 64;
// Up to kIndexLds rows whose ids fit a word beside the row's number are sorted in LDS in one launch; more
// by the launches of index_sort_* and index_words_*.  us, one launch / seven: 4096 rows 20.6 / 29.3, 7088 31.9 / 30.7, 9000 39.0 / 31.8.
constexpr int kIndexLds = 8192;

// Lanes of `active` whose low `bits` bits of d equal this lane's.
__device__ inline unsigned long long match_lanes(unsigned d, unsigned long long active) {
  unsigned long long m = active;
#pragma unroll
  for (int b = 0; b < 8; b++) {
    const bool bit = (d >> b) & 1;
    const unsigned long long v = __ballot(bit);
    m &= bit ? v : ~v;
  }
  return m;
}

// exclusive scan over the workgroup's 1024 values; `total`: their sum
__device__ inline unsigned block_scan(unsigned v, unsigned *wave_sums, unsigned *total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  unsigned incl = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned u = __shfl_up(incl, o, 64);
    if (lane >= o) incl += u;
  }
  if (lane == 63) wave_sums[wave] = incl;
  __syncthreads();
  unsigned base = 0, all = 0;
  for (int w = 0; w < kIndexWaves; w++) {
    const unsigned s = wave_sums[w];
    if (w < wave) base += s;
    all += s;
  }
  __syncthreads();
  *total = all;
  return base + incl - v;
}

// a row whose id is no whole number in [0, V) is a word of its own
__device__ inline unsigned word_key(float id, int V) {
  const int k = (int)id;
  return (id >= 0.f && id < (float)V && (float)k == id) ? k : V;
}

// One workgroup.  A row whose id is no whole number in [0, V) is a word of its own (key V).  What bounds
// it is the chain of sweeps (about 1 us each), not the work: every wavefront takes one stretch of the rows in
// order, so that ranks are stable without a second pass.
__global__ __launch_bounds__(kIndexThreads) void embed_index_kernel(int *__restrict__ index, float *__restrict__ ids_out,
                                                                    const float *__restrict__ x, const int *__restrict__ rows, int n, int V,
                                                                    int leaf_rows, int passes, int row_bits) {
  __shared__ unsigned lds[2 * kIndexLds];
  __shared__ unsigned hist[kIndexWaves][256];
  __shared__ unsigned wave_sums[kIndexWaves], first_sums[kIndexWaves], leaf_sums[kIndexWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const unsigned long long below = (1ull << lane) - 1;
  // row i: id key(i), vertex row val(i)
  unsigned *ka = lds, *kb = lds + kIndexLds;
  auto key = [&](int i) { return ka[i] >> row_bits; };
  auto val = [&](int i) { return ka[i] & ((1u << row_bits) - 1); };
  auto put = [&](unsigned *k, int i, unsigned id, unsigned row) { k[i] = id << row_bits | row; };
  int *slot = index + 4, *order = slot + n, *at = order + n;
  float *word = reinterpret_cast<float *>(at + n);
  const int per = ((n + kIndexWaves - 1) / kIndexWaves + 63) / 64 * 64;
  const int beg = min(n, wave * per), end = min(n, beg + per);

#pragma unroll 4
  for (int i = beg + lane; i < end; i += 64) {
    const float id = x[rows[i]];
    ids_out[i] = id;
    put(ka, i, word_key(id, V), i);
  }
  for (int pass = 0; pass < passes; pass++) {
    const int shift = 8 * pass;
    for (int i = tid; i < kIndexWaves * 256; i += kIndexThreads) (&hist[0][0])[i] = 0;
    __syncthreads();
    for (int i = beg + lane; i < end; i += 64) atomicAdd(&hist[wave][(key(i) >> shift) & 255], 1u);
    __syncthreads();
    {  // where the rows of a digit that a wavefront holds go: digits first, wavefronts within
      const int d = tid >> 2, w0 = (tid & 3) * 4;
      unsigned v[4], sum = 0, all;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        v[j] = sum;
        sum += hist[w0 + j][d];
      }
      const unsigned base = block_scan(sum, wave_sums, &all);
#pragma unroll
      for (int j = 0; j < 4; j++) hist[w0 + j][d] = base + v[j];
    }
    __syncthreads();
    for (int i0 = beg; i0 < end; i0 += 64) {
      const int i = i0 + lane;
      const bool in = i < end;
      const unsigned k = in ? key(i) : 0, v = in ? val(i) : 0, d = (k >> shift) & 255;
      const unsigned long long m = match_lanes(d, __ballot(in));
      if (in) {
        const int rank = __popcll(m & below);
        const unsigned pos = hist[wave][d] + rank;
        put(kb, pos, k, v);
        if ((m & ~below & ~(1ull << lane)) == 0) hist[wave][d] = pos + 1;  // (the last of its digit in this step)
      }
    }
    __syncthreads();
    unsigned *t = ka; ka = kb; kb = t;
  }
  // Segments of equal ids.  The words no inner vertex looked up come first (their rows of the f columns are
  // zero, as those of the leaves): rows of a segment ascend, so its last one tells.
  auto bounds = [&](int p, bool *first, bool *last, bool *leaves) {
    const unsigned k = key(p);
    *first = p == 0 || k == (unsigned)V || key(p - 1) != k;
    *last = p == n - 1 || k == (unsigned)V || key(p + 1) != k;
    *leaves = *last && (int)val(p) < leaf_rows;
  };
  unsigned nf = 0, nl = 0;
  for (int i0 = beg; i0 < end; i0 += 64) {
    bool f = false, l = false, z = false;
    if (i0 + lane < end) bounds(i0 + lane, &f, &l, &z);
    nf += __popcll(__ballot(f));
    nl += __popcll(__ballot(z));
  }
  if (lane == 0) first_sums[wave] = nf, leaf_sums[wave] = nl;
  __syncthreads();
  unsigned fbase = 0, zbase = 0, words = 0, leaf_words = 0;
  for (int w = 0; w < kIndexWaves; w++) {
    if (w < wave) fbase += first_sums[w], zbase += leaf_sums[w];
    words += first_sums[w];
    leaf_words += leaf_sums[w];
  }
  if (tid == 0) {
    index[0] = words;
    index[1] = leaf_words;
    index[2] = index[3] = 0;
  }
  unsigned *seg_slot = kb;
  for (int sweep = 0; sweep < 2; sweep++) {
    unsigned fcount = fbase, zcount = zbase;
    for (int i0 = beg; i0 < end; i0 += 64) {
      const int p = i0 + lane;
      bool f = false, l = false, z = false;
      if (p < end) bounds(p, &f, &l, &z);
      const unsigned long long fm = __ballot(f), zm = __ballot(z);
      const unsigned seg = fcount + __popcll(fm & (below | 1ull << lane)) - 1, leaves_before = zcount + __popcll(zm & below);
      fcount += __popcll(fm);
      zcount += __popcll(zm);
      if (p >= end) continue;
      const int row = val(p);
      if (sweep == 0) {
        if (l) {
          const unsigned s = z ? leaves_before : leaf_words + (seg - leaves_before);
          seg_slot[seg] = s;
          word[s] = ids_out[row];
        }
      } else {
        const int s = seg_slot[seg];
        slot[row] = s;
        order[p] = row;
        at[p] = s;
      }
    }
    __syncthreads();
  }
}

// The same over many workgroups: a launch per dependent step.  Workgroup g has one stretch of the rows (SortWork), its wavefronts
// parts of it in order; a digit's rows go behind those of the digits before and of the stretches before, both
// counted from the table of counts that the launch before left.  Bound by the launches, 5 us each: 16384 rows 33 us, 73000 37,
// 300000 55, where one workgroup, its rows in memory, took 65, 363 (540 inside a step) and 2090.
struct SortWork {
  unsigned *ka, *va, *kb, *vb;  // [n] ids and rows, from and to
  unsigned *counts;             // [groups][256] rows of a digit in a stretch (where the index goes afterwards)
  unsigned *words;              // [groups][2] words that begin in a stretch, words of leaves only (where the sort had its rows)
  int n, per, groups;           // rows of a stretch: a multiple of 1024
  __device__ inline void stretch(int *beg, int *end) const {
    const int own = per / kIndexWaves;
    *beg = min(n, (int)blockIdx.x * per + (int)(threadIdx.x >> 6) * own);
    *end = min(n, *beg + own);
  }
};
constexpr int kSortGroups = 256;
static int sort_per(int n) { return std::max(1, (n + kSortGroups * 1024 - 1) / (kSortGroups * 1024)) * 1024; }
static int sort_groups(int n) { return (n + sort_per(n) - 1) / sort_per(n); }

template <bool FIRST>
__global__ __launch_bounds__(kIndexThreads) void index_sort_count_kernel(SortWork s, float *__restrict__ ids_out, const float *__restrict__ x,
                                                                         const int *__restrict__ rows, int V, int shift) {
  __shared__ unsigned hist[256];
  if (threadIdx.x < 256) hist[threadIdx.x] = 0;
  __syncthreads();
  int beg, end;
  s.stretch(&beg, &end);
#pragma unroll 4
  for (int i = beg + (threadIdx.x & 63); i < end; i += 64) {
    unsigned k;
    if constexpr (FIRST) {
      const float id = x[rows[i]];
      ids_out[i] = id;
      k = word_key(id, V);
      s.ka[i] = k;
      s.va[i] = i;
    } else {
      k = s.ka[i];
    }
    atomicAdd(&hist[(k >> shift) & 255], 1u);
  }
  __syncthreads();
  if (threadIdx.x < 256) s.counts[blockIdx.x * 256 + threadIdx.x] = hist[threadIdx.x];
}

__global__ __launch_bounds__(kIndexThreads) void index_sort_place_kernel(SortWork s, int shift) {
  __shared__ unsigned hist[kIndexWaves][256];
  __shared__ unsigned wave_sums[kIndexWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = blockIdx.x;
  const unsigned long long below = (1ull << lane) - 1;
  int beg, end;
  s.stretch(&beg, &end);
  for (int i = tid; i < kIndexWaves * 256; i += kIndexThreads) (&hist[0][0])[i] = 0;
  const int d = tid >> 2, part = tid & 3;  // four lanes a digit
  unsigned all = 0, before = 0;
#pragma unroll 8
  for (int h = part; h < s.groups; h += 4) {
    const unsigned c = s.counts[h * 256 + d];
    all += c;
    before += h < g ? c : 0;
  }
  __syncthreads();
  for (int i = beg + lane; i < end; i += 64) atomicAdd(&hist[wave][(s.ka[i] >> shift) & 255], 1u);
  __syncthreads();
  {
    unsigned total;
    unsigned base = block_scan(all, wave_sums, &total);  // (of the digit's first lane: the digits before)
    base = __shfl(base, lane & ~3, 64);
#pragma unroll
    for (int o = 1; o < 4; o <<= 1) before += __shfl_xor(before, o, 64);
    unsigned v[4], sum = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      v[j] = sum;
      sum += hist[4 * part + j][d];
    }
    unsigned incl = sum;  // over the digit's four lanes
#pragma unroll
    for (int o = 1; o < 4; o <<= 1) {
      const unsigned u = __shfl_up(incl, o, 4);
      if (part >= o) incl += u;
    }
#pragma unroll
    for (int j = 0; j < 4; j++) hist[4 * part + j][d] = base + before + (incl - sum) + v[j];
  }
  __syncthreads();
  for (int i0 = beg; i0 < end; i0 += 64) {
    const int i = i0 + lane;
    const bool in = i < end;
    const unsigned k = in ? s.ka[i] : 0, v = in ? s.va[i] : 0, q = (k >> shift) & 255;
    const unsigned long long m = match_lanes(q, __ballot(in));
    if (in) {
      const unsigned pos = hist[wave][q] + __popcll(m & below);
      s.kb[pos] = k;
      s.vb[pos] = v;
      if ((m & ~below & ~(1ull << lane)) == 0) hist[wave][q] = pos + 1;  // (the last of its digit in this step)
    }
  }
}

// Segments of equal ids (s.ka, s.va: sorted), as in embed_index_kernel.  STEP 0: a stretch's words; 1: the words' places, by
// segment, in s.kb; 2: the words of the rows.
template <int STEP>
__global__ __launch_bounds__(kIndexThreads) void index_words_kernel(SortWork s, int *__restrict__ index, const float *__restrict__ ids, int V, int leaf_rows) {
  __shared__ unsigned own[kIndexWaves][2], others[kIndexWaves][4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = blockIdx.x, n = s.n;
  const unsigned long long below = (1ull << lane) - 1;
  unsigned *counts = s.words;
  int beg, end;
  s.stretch(&beg, &end);
  auto bounds = [&](int p, bool *first, bool *last, bool *leaves) {
    const unsigned k = s.ka[p];
    *first = p == 0 || k == (unsigned)V || s.ka[p - 1] != k;
    *last = p == n - 1 || k == (unsigned)V || s.ka[p + 1] != k;
    *leaves = *last && (int)s.va[p] < leaf_rows;
  };
  unsigned nf = 0, nl = 0;
  for (int i0 = beg; i0 < end; i0 += 64) {
    bool f = false, l = false, z = false;
    if (i0 + lane < end) bounds(i0 + lane, &f, &l, &z);
    nf += __popcll(__ballot(f));
    nl += __popcll(__ballot(z));
  }
  if (lane == 0) own[wave][0] = nf, own[wave][1] = nl;
  unsigned c[4] = {0, 0, 0, 0};  // words and words of leaves: of the stretches before, of all
  if (STEP > 0 && tid < s.groups) {
    c[2] = counts[2 * tid];
    c[3] = counts[2 * tid + 1];
    if (tid < g) c[0] = c[2], c[1] = c[3];
  }
#pragma unroll
  for (int j = 0; j < 4; j++) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) c[j] += __shfl_xor(c[j], o, 64);
    if (lane == 0) others[wave][j] = c[j];
  }
  __syncthreads();
  if constexpr (STEP == 0) {
    if (tid < 2) {
      unsigned sum = 0;
      for (int w = 0; w < kIndexWaves; w++) sum += own[w][tid];
      counts[2 * g + tid] = sum;
    }
    return;
  }
  unsigned fcount = 0, zcount = 0, words = 0, leaf_words = 0;
  for (int w = 0; w < kIndexWaves; w++) {
    fcount += others[w][0] + (w < wave ? own[w][0] : 0);
    zcount += others[w][1] + (w < wave ? own[w][1] : 0);
    words += others[w][2];
    leaf_words += others[w][3];
  }
  if (STEP == 1 && g == 0 && tid == 0) {
    index[0] = words;
    index[1] = leaf_words;
    index[2] = index[3] = 0;
  }
  int *slot = index + 4, *order = slot + n, *at = order + n;
  float *word = reinterpret_cast<float *>(at + n);
  for (int i0 = beg; i0 < end; i0 += 64) {
    const int p = i0 + lane;
    bool f = false, l = false, z = false;
    if (p < end) bounds(p, &f, &l, &z);
    const unsigned long long fm = __ballot(f), zm = __ballot(z);
    const unsigned seg = fcount + __popcll(fm & (below | 1ull << lane)) - 1, leaves_before = zcount + __popcll(zm & below);
    fcount += __popcll(fm);
    zcount += __popcll(zm);
    if (p >= end) continue;
    const int row = s.va[p];
    if constexpr (STEP == 1) {
      if (l) {
        const unsigned q = z ? leaves_before : leaf_words + (seg - leaves_before);
        s.kb[seg] = q;
        word[q] = ids[row];
      }
    } else {
      const int q = s.kb[seg];
      slot[row] = q;
      order[p] = row;
      at[p] = q;
    }
  }
}

// out[s] = the table row of word s
__global__ __launch_bounds__(256) void embed_words_kernel(float *__restrict__ out, int ld, const int *__restrict__ index, int n,
                                                          const float *__restrict__ table, int E) {
  const int s = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (s >= index[0]) return;
  const float id = reinterpret_cast<const float *>(index + 4 + 3 * (long)n)[s];
  const long off = (long)(int)(id * (float)E);
  for (int c = lane; c < E; c += 64) out[(long)s * ld + c] = off >= 0 ? table[off + c] : 0.f;
}

// table row of word s += dy[s]; words that are no whole number may share a row's elements
__global__ __launch_bounds__(256) void embed_words_bwd_kernel(float *__restrict__ dtable, const int *__restrict__ index, int n,
                                                              const float *__restrict__ dy, int ld, int E) {
  const int s = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (s >= index[0]) return;
  const long off = (long)(int)(reinterpret_cast<const float *>(index + 4 + 3 * (long)n)[s] * (float)E);
  if (off < 0) return;
  for (int c = lane; c < E; c += 64) unsafeAtomicAdd(dtable + off + c, dy[(long)s * ld + c]);
}

// dst[t] = src[slot[t]]: a wavefront a row; rows below head_rows only their first head_q float4
__global__ __launch_bounds__(256) void spread_rows_kernel(float4 *__restrict__ dst, long ld_dst, const float4 *__restrict__ src, long ld_src,
                                                          const int *__restrict__ slot, int n, int q, int head_rows, int head_q,
                                                          const float *__restrict__ ids, float *__restrict__ ids_out) {
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (t >= n) return;
  if (ids_out && lane == 0) ids_out[t] = ids[t];
  const float4 *s = src + slot[t] * ld_src;
  float4 *d = dst + t * ld_dst;
  const int end = t < head_rows ? head_q : q;
#pragma unroll 4
  for (int c = lane; c < end; c += 64) d[c] = s[c];
}

// Sums over the sorted rows, in pieces of a few rows that do not follow the segments: however often a word
// occurs, the work per wavefront is the same.  A wavefront takes one piece of 256 columns.  A segment that
// lies inside a piece is stored; the part of one that crosses a border goes to `part`: row 2c the
// part that began in an earlier piece, row 2c + 1 the one that goes on in the next (a segment that
// does both: row 2c).
// Pieces of 16 rows (one batch of loads) while they are few, else of 64 (2368 x 2048: 13.3 us in pieces of 64).
// TOTALS: the sum of all of a piece's rows to row c of `totals` as well: what is left to read for the sum of all rows is a
// sixteenth or less of them (73000 rows of 4096: 321 -> 323 us here, the bias's own pass over them 239 -> 15).
constexpr int kSumFew = 8192;
static int sum_rows(int n) { return n <= kSumFew ? 16 : 64; }
template <int kSumRows, bool TOTALS>
__global__ __launch_bounds__(256) void gather_sums_kernel(float *__restrict__ dst, long ld_dst, const float *__restrict__ src, long ld_src,
                                                          const int *__restrict__ order, const int *__restrict__ at, int n, int w,
                                                          float *__restrict__ part, float *__restrict__ totals) {
  const int lane = threadIdx.x & 63, c = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int p0 = c * kSumRows, count = min(kSumRows, n - p0), col = blockIdx.y * 256 + 4 * lane;
  if (count <= 0) return;
  const int row = lane < count ? order[p0 + lane] : 0, slot = lane < count ? at[p0 + lane] : -1;
  const int before = p0 > 0 ? at[p0 - 1] : -1, after = p0 + count < n ? at[p0 + count] : -1;
  const bool in = col < w;
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f), all = acc;
  int cur = __builtin_amdgcn_readlane(slot, 0);
  auto put = [&](float *to) {
    if (in) *reinterpret_cast<float4 *>(to + col) = acc;
    if (TOTALS) all.x += acc.x, all.y += acc.y, all.z += acc.z, all.w += acc.w;
    acc = make_float4(0.f, 0.f, 0.f, 0.f);
  };
  constexpr int U = 16;
  for (int i = 0; i < count; i += U) {
    float4 v[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (i + u < count && in) v[u] = *reinterpret_cast<const float4 *>(src + __builtin_amdgcn_readlane(row, i + u) * ld_src + col);
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (i + u >= count) break;
      const int s = __builtin_amdgcn_readlane(slot, i + u);
      if (s != cur) {
        put(cur == before ? part + (long)2 * c * w : dst + cur * ld_dst);
        cur = s;
      }
      acc.x += v[u].x, acc.y += v[u].y, acc.z += v[u].z, acc.w += v[u].w;
    }
  }
  if (cur == before) put(part + (long)2 * c * w);
  else if (cur == after) put(part + (long)(2 * c + 1) * w);
  else put(dst + cur * ld_dst);
  if (TOTALS && in) *reinterpret_cast<float4 *>(totals + (long)c * w + col) = all;
}

// The segments that cross borders: the workgroup of the piece where one begins adds up its parts, a
// quarter of them to a wavefront, in order.
template <int kSumRows>
__global__ __launch_bounds__(256) void gather_sums_across_kernel(float *__restrict__ dst, long ld_dst, const int *__restrict__ at, int n, int w,
                                                                 const float *__restrict__ part) {
  __shared__ float4 sums[4][64];
  const int c = blockIdx.x, p1 = (c + 1) * kSumRows, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (p1 >= n) return;
  const int s = at[p1];
  if (at[p1 - 1] != s || (c > 0 && at[c * kSumRows - 1] == s)) return;  // nothing crosses here, or it began earlier
  // pieces c + 1 .. last hold the rest of it
  int last = c + 1;
  for (;;) {
    const int p = (last + lane + 1) * kSumRows;  // the first row behind piece last + lane
    const unsigned long long stops = __ballot(p >= n || at[min(p, n - 1)] != s);
    if (stops) {
      last += __ffsll(stops) - 1;
      break;
    }
    last += 64;
  }
  const int parts = last - c + 1, per = (parts + 3) / 4, a = wave * per, b = min(parts, a + per), col = blockIdx.y * 256 + 4 * lane;
  const bool in = col < w;
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  constexpr int U = 8;
  for (int i = a; i < b; i += U) {
    float4 v[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (i + u < b && in) v[u] = *reinterpret_cast<const float4 *>(part + (long)(i + u == 0 ? 2 * c + 1 : 2 * (c + i + u)) * w + col);
    }
#pragma unroll
    for (int u = 0; u < U; u++) acc.x += v[u].x, acc.y += v[u].y, acc.z += v[u].z, acc.w += v[u].w;
  }
  sums[wave][lane] = acc;
  __syncthreads();
  if (wave == 0 && in) {
#pragma unroll
    for (int q = 1; q < 4; q++) {
      const float4 v = sums[q][lane];
      acc.x += v.x, acc.y += v.y, acc.z += v.z, acc.w += v.w;
    }
    *reinterpret_cast<float4 *>(dst + s * ld_dst + col) = acc;
  }
}

}  // namespace cavs

using namespace cavs;

extern "C" {

size_t cavs_embed_index_ints(int n) { return 4 + 4 * (size_t)std::max(n, 0); }

size_t cavs_embed_index_workspace(int n) { return 4 * sizeof(unsigned) * (size_t)std::max(n, 0); }

int cavs_embed_index(int *index, float *ids_out, const float *x, const int *rows, int n, int V, int leaf_rows, void *workspace,
                     size_t workspace_bytes, void *stream) {
  CAVS_REQUIRE(n >= 0 && n < (1 << 27) && V > 0 && V < (1 << 24), "cavs_embed_index: bad shape n=%d V=%d", n, V);
  CAVS_REQUIRE(index, "cavs_embed_index: null pointer");
  CAVS_REQUIRE(n == 0 || (ids_out && x && rows), "cavs_embed_index: null pointer");
  const size_t need = cavs_embed_index_workspace(n);
  CAVS_REQUIRE(need == 0 || (workspace && workspace_bytes >= need), "cavs_embed_index: workspace of %zu bytes needed, %zu given", need, workspace_bytes);
  const int passes = V < (1 << 8) ? 1 : V < (1 << 16) ? 2 : 3;  // (keys 0 .. V)
  hipStream_t st = as_stream(stream);
  int row_bits = 8;  // (up to 256 rows: any id a float counts to)
  while ((1 << row_bits) < std::min(n, kIndexLds)) row_bits++;
  if (n <= kIndexLds && (n <= 256 || V < 1 << (32 - row_bits))) {  // (ids 0 .. V)
    launch(embed_index_kernel, 1, kIndexThreads, 0, st, index, ids_out, x, rows, n, V, leaf_rows, passes, row_bits);
    CAVS_LAUNCH_CHECK();
    return CAVS_OK;
  }
  unsigned *w = static_cast<unsigned *>(workspace);
  SortWork s{w, w + n, w + 2 * (size_t)n, w + 3 * (size_t)n, reinterpret_cast<unsigned *>(index + 4), nullptr, n, sort_per(n), sort_groups(n)};
  for (int pass = 0; pass < passes; pass++) {
    if (pass == 0) launch(index_sort_count_kernel<true>, s.groups, kIndexThreads, 0, st, s, ids_out, x, rows, V, 0);
    else launch(index_sort_count_kernel<false>, s.groups, kIndexThreads, 0, st, s, nullptr, nullptr, nullptr, V, 8 * pass);
    launch(index_sort_place_kernel, s.groups, kIndexThreads, 0, st, s, 8 * pass);
    std::swap(s.ka, s.kb);
    std::swap(s.va, s.vb);
  }
  s.words = s.vb;
  launch(index_words_kernel<0>, s.groups, kIndexThreads, 0, st, s, index, ids_out, V, leaf_rows);
  launch(index_words_kernel<1>, s.groups, kIndexThreads, 0, st, s, index, ids_out, V, leaf_rows);
  launch(index_words_kernel<2>, s.groups, kIndexThreads, 0, st, s, index, ids_out, V, leaf_rows);
  CAVS_LAUNCH_CHECK();
  return CAVS_OK;
}

int cavs_embed_words(float *out, int ld_out, const int *index, const float *table, int n, int E, void *stream) {
  CAVS_REQUIRE(n >= 0 && E > 0 && ld_out >= E, "cavs_embed_words: bad shape n=%d E=%d ld=%d", n, E, ld_out);
  if (n == 0) return CAVS_OK;
  CAVS_REQUIRE(out && index && table, "cavs_embed_words: null pointer");
  launch(embed_words_kernel, (n + 3) / 4, 256, 0, as_stream(stream), out, ld_out, index, n, table, E);
  CAVS_LAUNCH_CHECK();
  return CAVS_OK;
}

int cavs_embed_words_bwd(float *dtable, const int *index, const float *dy, int ld_dy, int n, int E, void *stream) {
  CAVS_REQUIRE(n >= 0 && E > 0 && ld_dy >= E, "cavs_embed_words_bwd: bad shape n=%d E=%d ld=%d", n, E, ld_dy);
  if (n == 0) return CAVS_OK;
  CAVS_REQUIRE(dtable && index && dy, "cavs_embed_words_bwd: null pointer");
  launch(embed_words_bwd_kernel, (n + 3) / 4, 256, 0, as_stream(stream), dtable, index, n, dy, ld_dy, E);
  CAVS_LAUNCH_CHECK();
  return CAVS_OK;
}

int cavs_spread_rows(float *dst, int ld_dst, const float *src, int ld_src, const int *index, int n, int w, int head_rows, int head_w,
                     const float *ids, float *ids_out, void *stream) {
  CAVS_REQUIRE(n >= 0 && w >= 0 && w % 4 == 0 && head_w >= 0 && head_w <= w && head_w % 4 == 0 && ld_dst >= w && ld_src >= w && ld_dst % 4 == 0 &&
                   ld_src % 4 == 0,
               "cavs_spread_rows: bad shape n=%d w=%d head_w=%d ld=%d,%d", n, w, head_w, ld_dst, ld_src);
  if (n == 0 || w == 0) return CAVS_OK;
  CAVS_REQUIRE(dst && src && index && aligned16(dst) && aligned16(src), "cavs_spread_rows: null or misaligned pointer");
  launch(spread_rows_kernel, (n + 3) / 4, 256, 0, as_stream(stream), reinterpret_cast<float4 *>(dst), ld_dst / 4,
         reinterpret_cast<const float4 *>(src), ld_src / 4, index + 4, n, w / 4, head_rows, head_w / 4, ids,
         ids ? ids_out : nullptr);
  CAVS_LAUNCH_CHECK();
  return CAVS_OK;
}

size_t cavs_gather_sums_workspace(int n, int w) {
  if (n <= 0 || w <= 0) return 0;
  // (no less than for any smaller n)
  return 2 * sizeof(float) * (size_t)std::max((n + sum_rows(n) - 1) / sum_rows(n), (std::min(n, kSumFew) + 15) / 16) * w;
}

int cavs_gather_sums(float *dst, int ld_dst, const float *src, int ld_src, const int *index, int n, int w, void *workspace,
                     size_t workspace_bytes, void *stream) {
  return cavs_gather_sums_totals(dst, ld_dst, src, ld_src, index, n, w, nullptr, workspace, workspace_bytes, stream);
}

int cavs_gather_sums_pieces(int n) { return n > 0 ? (n + sum_rows(n) - 1) / sum_rows(n) : 0; }

int cavs_gather_sums_totals(float *dst, int ld_dst, const float *src, int ld_src, const int *index, int n, int w, float *totals, void *workspace,
                            size_t workspace_bytes, void *stream) {
  CAVS_REQUIRE(n >= 0 && w >= 0 && w % 4 == 0 && ld_dst >= w && ld_src >= w && ld_dst % 4 == 0 && ld_src % 4 == 0,
               "cavs_gather_sums: bad shape n=%d w=%d ld=%d,%d", n, w, ld_dst, ld_src);
  if (n == 0 || w == 0) return CAVS_OK;
  CAVS_REQUIRE(dst && src && index && aligned16(dst) && aligned16(src) && (!totals || aligned16(totals)), "cavs_gather_sums: null or misaligned pointer");
  const size_t need = cavs_gather_sums_workspace(n, w);
  CAVS_REQUIRE(workspace && workspace_bytes >= need && aligned16(workspace), "cavs_gather_sums: workspace of %zu bytes needed, %zu given", need, workspace_bytes);
  const int per = sum_rows(n), pieces = (n + per - 1) / per, cols = (w + 255) / 256;
  const int *order = index + 4 + n, *at = order + n;
  float *part = static_cast<float *>(workspace);
  hipStream_t st = as_stream(stream);
  launch(per == 16 ? totals ? gather_sums_kernel<16, true> : gather_sums_kernel<16, false> : totals ? gather_sums_kernel<64, true> : gather_sums_kernel<64, false>,
         dim3((pieces + 3) / 4, cols), 256, 0, st, dst, ld_dst, src, ld_src, order, at, n, w, part, totals);
  CAVS_LAUNCH_CHECK();
  if (pieces > 1) {
    launch(per == 16 ? gather_sums_across_kernel<16> : gather_sums_across_kernel<64>, dim3(pieces - 1, cols), 256, 0, st, dst, ld_dst, at, n, w, part);
    CAVS_LAUNCH_CHECK();
  }
  return CAVS_OK;
}

}  // extern "C"
