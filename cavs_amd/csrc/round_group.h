// Rounds of a batch in one launch per direction for all three vertex functions and every hidden size
// of whole tiles up to 512: the construction of round_tail.hip (trees of the message flow dealt to
// groups of workgroups that share an XCD's L2, weights in registers for the whole launch, one barrier
// per round inside the group) without what ties that one to H = 512 and to the Tree-LSTM.
//
// What bounds a round here is latency.  As a launch of its own a round costs 4.4 to 6 us however small it
// is; here it is the L2 round trips of the barrier and of the operand rows plus the products.  So:
//   * a group is the H / 16 workgroups of 16 hidden units each -- the fewest whose registers hold the
//     weights -- and as many groups share an XCD as its 32 CUs give room for (one at H = 512, four at
//     H = 128): fewer rows per group is fewer tiles per round;
//   * everything a round needs to know about its rows (children, destinations) comes in one record of
//     32 bytes per row, built on the host and fetched a round ahead: no chain of index loads
//     stands between two rounds;
//   * the plan is read from memory, so a launch runs any number of rounds (chains of hundreds).
// A wavefront owns ceil(H / 128) k-groups of 16 of its workgroup's columns; those beyond H are dropped.
#pragma once
#include <algorithm>
#include <type_traits>

#include "round_sync.h"

namespace cavs {

constexpr int kGroupMaxH = 512;
constexpr int kGroupRows = 32;    // rows per list: eight tiles of four
constexpr int kGroupWgsPerXcd = 32;
// Dynamic LDS of every launch: more than half of a CU's 160 KB, so that workgroups land one to a CU.
constexpr size_t kGroupLds = 84 << 10;

enum { GROUP_TREELSTM = 0, GROUP_LSTM = 1, GROUP_TREEFC = 2 };

struct GroupPlan {
  const int4 *groups;  // [ngroups] first list, lists, arrivals
  const int4 *lists;   // [*] first record, rows, arrivals to wait for; 1: it arrives, + 2 (backward): rows without a parent
  const int4 *recs;    // [*][2]
  unsigned *sync;
  int ngroups, wgs, spin_max, expect;
  bool whole_lines;  // of the rows the launch writes and reads (ld_row)
  bool wide;         // tiles of sixteen rows
};

template <int I, int N, class F>
__device__ inline void unrolled(F &&f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    unrolled<I + 1, N>(f);
  }
}

// A row of the plan by the scalar unit: nothing in the launch writes it, but the compiler cannot know that, and a
// vector load here would be waited for together with the stores of the list before.
__device__ inline int4 plan_row(const int4 *p) {
  typedef int i4 __attribute__((ext_vector_type(4)));
  const i4 v = *(const __attribute__((address_space(4))) i4 *)p;
  return int4{v[0], v[1], v[2], v[3]};
}

// A load is waited for here: the wait behind a branch further down would be for everything that may be under way by then
__device__ inline void arrived(float v) { asm volatile("" ::"v"(v)); }
// row * ld floats behind p: one multiplication of 32 bits (row >= 0)
template <class T>
__device__ inline T *row_at(T *p, int row, unsigned ld) { return p + (size_t)(unsigned)row * ld; }

// What every list of a launch goes through besides its products: the plan, the records of the next
// list on their way while this one runs, and the group's barrier.
struct GroupWalk {
  const int4 *lists, *recs;
  unsigned *status, *gsync;
  int nlists, ct;
  unsigned arrived;
  int4 cur, nxt, ahead, rec;
  unsigned words;  // the group's, as they were when the list began
  bool first_wait;
  __device__ inline bool start(const GroupPlan &p, int4 (*s_rec)[2 * kGroupRows], int *s_bail) {
    const int idx = blockIdx.x >> 3, grp = (blockIdx.x & 7) + 8 * (idx / p.wgs);  // workgroup b sits on XCD b % 8
    ct = idx % p.wgs;
    if (grp >= p.ngroups) return false;
    const int4 g = plan_row(p.groups + grp);
    nlists = g.y;
    if (nlists == 0) return false;
    status = p.sync + TAIL_STATUS;
    gsync = p.sync + TAIL_GROUP_WORDS * (grp + 1);
    // (an earlier launch on this block gave up and nobody has cleared it: nothing here can be trusted)
    if (__hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) return false;
    lists = p.lists + g.x;
    recs = p.recs;
    arrived = 0;
    first_wait = true;
    if (threadIdx.x == 0) *s_bail = 0;
    cur = plan_row(lists);
    nxt = plan_row(lists + (nlists > 1 ? 1 : 0));
    put(s_rec[0], cur, record(cur));
    if (threadIdx.x == 0) __hip_atomic_fetch_or(gsync + TAIL_XCC, 1u << xcc_id(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
  }
  // half a record to a thread, the same to every wavefront (of a row beyond the list's: its first row's)
  __device__ inline int4 record(const int4 &list) const {
    const int i = (threadIdx.x & 63) >> 1;
    return recs[2L * (list.x + (i < list.y ? i : 0)) + (threadIdx.x & 1)];
  }
  __device__ inline void put(int4 *to, const int4 &list, const int4 &v) const {
    if (threadIdx.x < 2 * kGroupRows) to[threadIdx.x] = (int)(threadIdx.x >> 1) < list.y ? v : int4{-1, -1, -1, -1};
  }
  // A list begins: the group's words, then what its gate functions and the lists behind it read of the launches before.  Loads come
  // back in the order they were made, and those go to memory: with the words behind them, the words were another trip; so they are asked
  // for first and looked at when the addresses are done.  Nothing here is conditional, or the waits, which then have to hold for
  // either way, would be for everything: a wavefront without rows asks for what the list's first needs.
  // Cycles from list to list, 16 chains of 20, H = 128: 4200 forward and 3850 backward -> 3550 and 3250 (with the last tile of a list by
  // itself: 300 of them).  Passes of 16 steps: those chains 2527 -> 2430 us, Tree-FC, 64 trees, H = 256 2152 -> 1968; 37 chains,
  // H = 200, one step with its gradients 635 -> 616.
  __device__ inline void begin(const GroupPlan &p, int r) {
    words = tail_ask(gsync, p.expect);
    ahead = lists[r + 2 < nlists ? r + 2 : nlists - 1];  // (not by the scalar unit: waits for LDS would be for it too)
    rec = record(nxt);
  }
  // (where there is nothing to wait for, the barrier at the end of the list before is enough; a wait that gives up
  // sets *s_bail, looked at behind the barrier that completes the partial sums)
  __device__ inline void wait(const GroupPlan &p, int *s_bail) {
    if (cur.z <= 0) return;
    if (first_wait || !p.whole_lines || !__all(words >= (unsigned)cur.z))
      tail_wait(status, gsync, (unsigned)cur.z, p.expect, p.spin_max, first_wait, p.whole_lines, s_bail);
    asm volatile("" ::: "memory");  // (what the others wrote is read after this)
    first_wait = false;
  }
  // before the barrier that completes the list's partial sums
  __device__ inline void keep_next(int r, int4 (*s_rec)[2 * kGroupRows]) const { put(s_rec[(r + 1) & 1], nxt, rec); }
  __device__ inline void done() {
    if (cur.w & 1) tail_arrive(gsync, ct, ++arrived);
    else __syncthreads();
  }
  __device__ inline void advance() {
    cur = nxt;
    nxt = int4{__builtin_amdgcn_readfirstlane(ahead.x), __builtin_amdgcn_readfirstlane(ahead.y), __builtin_amdgcn_readfirstlane(ahead.z),
               __builtin_amdgcn_readfirstlane(ahead.w)};
  }
};

// Parks the wavefront's four-row sums of NP products for tile t: [tile][wavefront][product][row][column].
template <int NP>
__device__ inline void group_park(float *red, const SlotSums<NP> &s, int t, int ks, int slot, int x) {
  float *dst = red + ((t * 8 + ks) * (NP * 4)) * 16 + x;
#pragma unroll
  for (int p = 0; p < NP; p++) dst[(p * 4 + slot) * 16] = s.r[p][0];
}
// product p of this thread's element (tile = wavefront, row = lane / 16), added up in wavefront order
template <int NP>
__device__ inline void group_sum(const float *red, int ks, int slot, int x, float (&v)[NP]) {
  const float *pre = red + (ks * 8 * (NP * 4) + slot) * 16 + x;
#pragma unroll
  for (int p = 0; p < NP; p++) {
    float s = 0.f;
#pragma unroll
    for (int g = 0; g < 8; g++) s += pre[(g * NP * 4 + p * 4) * 16];
    v[p] = s;
  }
}

// record of a row: {slab row, pool row of child 0, of child 1, pool row its message goes to}, {row of graph_out, ...}
struct GroupFwdArgs {
  float *pool;         // [*, MW]
  const float *xW;     // [N, ld_xw]: x * W; Tree-FC: the vertex input's rows (may be null)
  long ld_xw;
  const float *Wp;     // tile-major weights
  const float *bias;   // Tree-FC: may be null
  float *G, *hlr, *gates, *msg, *go;  // whole-batch slabs (msg, go may be null where the function allows)
  int H, act;
  GroupPlan plan;
  bool x_by_vertex;    // Tree-FC: xW in the order of graph_out
};

// record of a row: {slab row, slab rows of its two children, row of dret of child 0}, {that of child 1, ...}
struct GroupBwdArgs {
  float *dA;            // [N, ld]: d(x W) of the LSTMs, dz of Tree-FC
  long ld;
  float *dF, *dc;       // Tree-LSTM [2N, H]; [N, H]
  const float *WTp;     // tile-major transposed weights
  const float *gates, *G, *h, *dret;
  int H, leaf_rows, act;
  GroupPlan plan;
};

}  // namespace cavs

namespace cavs {
// mask: 0 or -1, made where the compiler cannot see which (an empty asm): of values that have just been loaded it would make a
// select with branches
__device__ inline float4 and4(int mask, const float4 &v) {
  return make_float4(__int_as_float(__float_as_int(v.x) & mask), __int_as_float(__float_as_int(v.y) & mask), __int_as_float(__float_as_int(v.z) & mask),
                     __int_as_float(__float_as_int(v.w) & mask));
}
__device__ inline float4 sel4(bool on, const float4 &v) { return on ? v : zero4(); }
}  // namespace cavs

#include "round_wide.h"

namespace cavs {

// ------------------------------------------------------------------ forward
// WIDE: tiles of sixteen rows (round_wide.h) where a list has them, four-row tiles for the rest.
template <int MODEL, int GPW, bool WIDE>
__global__ __launch_bounds__(512, 1) void group_fwd_kernel(GroupFwdArgs a) {
  constexpr int NP = MODEL == GROUP_TREELSTM ? 5 : MODEL == GROUP_LSTM ? 4 : 2, NW = MODEL == GROUP_TREEFC ? 2 : 4;
  constexpr int NC = MODEL == GROUP_LSTM ? 1 : 2;
  extern __shared__ __attribute__((aligned(16))) float red[];  // (16-byte accesses to an odd base are four times slower)
  __shared__ int4 s_rec[2][2 * kGroupRows];
  __shared__ int s_bail;
  GroupWalk w;
  if (!w.start(a.plan, s_rec, &s_bail)) return;
  const int H = a.H, KG = H / 16, tid = threadIdx.x, lane = tid & 63, ks = tid >> 6;
  const int x = lane & 15, slot = lane >> 4, j0 = w.ct * 16, ej = j0 + x;
  const long MW = MODEL == GROUP_TREEFC ? H : 2L * H;

  // this wavefront's weights: k-groups ks * GPW .. of column tile ct
  float4 wt[NW][GPW];
#pragma unroll
  for (int g = 0; g < GPW; g++) {
    const int kg = ks * GPW + g;
    const bool on = kg < KG;
    const float4 *base = reinterpret_cast<const float4 *>(a.Wp) + slot * 16 + x;
    const long k = on ? kg : 0;
#pragma unroll
    for (int q = 0; q < NW; q++) {
      long at;
      if constexpr (MODEL == GROUP_TREELSTM)  // U_iou [H, 3H], then U_f [H, H]
        at = q < 3 ? (k * 3 * KG + q * KG + w.ct) * 64 : 3L * H * H / 4 + (k * KG + w.ct) * 64;
      else if constexpr (MODEL == GROUP_LSTM)  // W' [H, 4H]
        at = (k * 4 * KG + q * KG + w.ct) * 64;
      else  // W [2H, H]: the left child's rows, then the right child's
        at = ((q * KG + k) * KG + w.ct) * 64;
      wt[q][g] = sel4(on, base[at]);
    }
  }
  if (ks < 4) __builtin_amdgcn_s_setprio(2);  // (wavefronts w and w + 4 share a SIMD: one goes first, see round_tail.hip)
  float bias[4] = {0.f, 0.f, 0.f, 0.f};
  if (MODEL != GROUP_TREEFC || a.bias) {
#pragma unroll
    for (int k = 0; k < (MODEL == GROUP_TREEFC ? 1 : 4); k++) bias[k] = a.bias[k * H + ej];
  }
  // where this lane's float4 of an operand row is (CAVS_MMA4's layout); lanes of k-groups beyond the wavefront's read the row's start and
  // drop it (their weights are zero, but zero times an infinity is a NaN)
  const int og = (lane >> 2) & 3, okg = ks * GPW + og;
  const bool inside = og < GPW && okg < KG;
  const int ka = inside ? 16 * okg + 4 * slot : 0;
  WideFwd<MODEL, GPW> wide(a, __builtin_amdgcn_readfirstlane(ks), lane, red);
  bool begun = false;  // (WIDE) the first tile's rows have been asked for
  __syncthreads();

  const float *x_rows = MODEL == GROUP_TREEFC && !a.xW ? a.Wp : a.xW;
  const unsigned x_ld = MODEL == GROUP_TREEFC && !a.xW ? 0 : (unsigned)a.ld_xw;
  for (int r = 0; r < w.nlists; r++) {
    const int4 *rt = s_rec[r & 1];
    const int n = w.cur.y < kGroupRows ? w.cur.y : kGroupRows, T = (n + 3) >> 2, TW = WIDE ? wide_tiles(n) : 0;
    w.begin(a.plan, r);
    // what does not depend on the rounds before (a wavefront without rows reads the first one's: see begin())
    const int eb = 4 * ks + slot;
    const bool eon = eb < n;
    int4 rec = rt[eon ? 2 * eb : 0];
    const int e_out = a.go && eon ? rt[2 * eb + 1].x : -1;
    float xw[4] = {0.f, 0.f, 0.f, 0.f};
    {
      const int row = MODEL == GROUP_TREEFC && a.x_by_vertex ? rt[eon ? 2 * eb + 1 : 1].x : rec.x;
      const float *p = row_at(x_rows, max(row, 0), x_ld) + ej;
#pragma unroll
      for (int k = 0; k < (MODEL == GROUP_TREEFC ? 1 : 4); k++) xw[k] = p[k * H];
    }
    if (!eon) rec = int4{-1, -1, -1, -1};

    // Operand rows, one float4 per child and tile, unconditionally (a missing child reads weights and is
    // masked); the next tile's are on their way while a tile is multiplied.
    struct Opnd {
      float4 v[NC];
      bool on[NC];
    };
    const float *at[NC], *kid[NC];
    auto rows = [&](int t, Opnd &o) {
      const int4 c = rt[2 * (4 * t + (lane & 3))];
#pragma unroll
      for (int k = 0; k < NC; k++) {
        const int row = k == 0 ? c.y : c.z;
        o.on[k] = row >= 0 && inside;
        at[k] = (row >= 0 ? row_at(a.pool, row, MW) : a.Wp) + ka;
      }
    };
    auto fetch = [&](Opnd &o) {
#pragma unroll
      for (int k = 0; k < NC; k++) o.v[k] = ld4(at[k]);
    };
    auto multiply = [&](int t, const Opnd &o) {
      floatx4 acc[NP];
#pragma unroll
      for (int p = 0; p < NP; p++) acc[p] = floatx4{0.f, 0.f, 0.f, 0.f};
      const float4 A = sel4(o.on[0], o.v[0]), B = NC == 2 ? sel4(o.on[NC - 1], o.v[NC - 1]) : zero4();
      const float4 S = make_float4(A.x + B.x, A.y + B.y, A.z + B.z, A.w + B.w);
      unrolled<0, GPW>([&](auto gc) {
        constexpr int g = decltype(gc)::value;
#pragma unroll
        for (int c = 0; c < 4; c++) {
          if constexpr (MODEL == GROUP_TREELSTM) {
            acc[0] = mma4<g>(elem(S, c), elem(wt[0][g], c), acc[0]);
            acc[1] = mma4<g>(elem(S, c), elem(wt[1][g], c), acc[1]);
            acc[2] = mma4<g>(elem(S, c), elem(wt[2][g], c), acc[2]);
            acc[3] = mma4<g>(elem(A, c), elem(wt[3][g], c), acc[3]);
            acc[4 % NP] = mma4<g>(elem(B, c), elem(wt[3][g], c), acc[4 % NP]);
          } else if constexpr (MODEL == GROUP_LSTM) {
#pragma unroll
            for (int q = 0; q < 4; q++) acc[q % NP] = mma4<g>(elem(A, c), elem(wt[q % NW][g], c), acc[q % NP]);
          } else {
            acc[0] = mma4<g>(elem(A, c), elem(wt[0][g], c), acc[0]);
            acc[1] = mma4<g>(elem(B, c), elem(wt[1][g], c), acc[1]);
          }
        }
      });
      SlotSums<NP> sums;
      sums.take(acc);
      sums.all();
      group_park<NP>(red, sums, t, ks, slot, x);
    };
    Opnd o, nx;
    const bool fours = 4 * TW < T;
    if (fours) rows(4 * TW, o);
#pragma unroll
    for (int k = 0; k < NC; k++) {  // the element's children
      const int row = k == 0 ? rec.y : rec.z;
      kid[k] = (row >= 0 ? row_at(a.pool, row, MW) : a.Wp) + ej;
    }
    w.wait(a.plan, &s_bail);
    if (WIDE && TW > 0 && !begun) wide.fetch(a, rt, n, 0, MW);
    if (fours) fetch(o);
    float e_h[NC], e_c[NC];
#pragma unroll
    for (int k = 0; k < NC; k++) {
      e_h[k] = ld_row(kid[k]);
      e_c[k] = MODEL != GROUP_TREEFC ? ld_row(kid[k] + H) : 0.f;
    }
    if constexpr (WIDE)
      for (int t = 0; t < TW; t++) wide.tile(a, rt, n, t, t + 1 < TW, MW, wt, red);
    if (fours) {
      for (int t = 4 * TW; t + 1 < T; t++) {
        rows(t + 1, nx);
        fetch(nx);
        multiply(t, o);
        o = nx;
      }
      multiply(T - 1, o);  // (by itself: in the loop it would wait for a fetch of its own successor)
    }
    arrived(MODEL != GROUP_TREEFC ? e_c[NC - 1] : e_h[NC - 1]);
    w.keep_next(r, s_rec);
    __syncthreads();
    if (s_bail) return;
    // a list that waits for nothing reads what this one could: its rows come while this one's gates are worked out
    if constexpr (WIDE) {
      begun = r + 1 < w.nlists && w.nxt.z <= 0 && wide_tiles(w.nxt.y) > 0;
      if (begun) wide.fetch(a, s_rec[(r + 1) & 1], w.nxt.y < kGroupRows ? w.nxt.y : kGroupRows, 0, MW);
    }

#pragma unroll
    for (int k = 0; k < NC; k++) {
      const bool on = (k == 0 ? rec.y : rec.z) >= 0;
      e_h[k] = on ? e_h[k] : 0.f;
      e_c[k] = on ? e_c[k] : 0.f;
    }
    float st[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, h = 0.f, cc = 0.f;  // what the backward pass wants, and the state
    const bool whole = w.cur.w & 4;
    if (eon) {
      float v[NP];
      if (WIDE && ks < 4 * TW) wide_sum<NP>(red, ks, lane, v);
      else group_sum<NP>(red, ks, slot, x, v);
      if constexpr (MODEL == GROUP_TREELSTM) {
        const TreeLstmCell q = whole ? treelstm_cell<true>(xw, v, bias, e_c[0], e_c[NC - 1]) : treelstm_cell(xw, v, bias, e_c[0], e_c[NC - 1]);
        st[0] = q.i; st[1] = q.o; st[2] = q.u; st[3] = q.f_l; st[4] = q.f_r; st[5] = q.tc;
        h = q.h; cc = q.c;
      } else if constexpr (MODEL == GROUP_LSTM) {
        const LstmCell q = whole ? lstm_cell<true>(xw, v, bias, e_c[0]) : lstm_cell(xw, v, bias, e_c[0]);
        st[0] = q.i; st[1] = q.f; st[2] = q.u; st[3] = q.o; st[4] = q.tc;
        h = q.h; cc = q.c;
      } else {
        float t = v[0] + v[1];
        if (a.bias) t += bias[0];
        if (a.xW) t += xw[0];
        h = !a.act ? (t > 0.f ? t : 0.f) : whole ? tanhf(t) : tanh_r(t);
      }
      // the message first: it is all a later round of this launch reads
      if (rec.w >= 0) {
        a.pool[rec.w * MW + ej] = h;
        if (MODEL != GROUP_TREEFC) a.pool[rec.w * MW + H + ej] = cc;
      }
    }
    w.done();
    if (eon) {  // what the backward pass and the caller read: on its way while the next round starts
      const long b = rec.x;
      if constexpr (MODEL != GROUP_TREEFC) {
        constexpr int NG = MODEL == GROUP_TREELSTM ? 6 : 5;
        float *g = a.gates + b * NG * H + ej;
#pragma unroll
        for (int k = 0; k < NG; k++) g[(long)k * H] = st[k];
      }
      if (a.msg) {
        a.msg[b * MW + ej] = h;
        if (MODEL != GROUP_TREEFC) a.msg[b * MW + H + ej] = cc;
      }
      if (e_out >= 0) a.go[(long)e_out * H + ej] = h;
      float *gp = a.G + b * NC * MW + ej;
#pragma unroll
      for (int k = 0; k < NC; k++) {
        gp[k * MW] = e_h[k];
        if (MODEL != GROUP_TREEFC) gp[k * MW + H] = e_c[k];
      }
      if constexpr (MODEL == GROUP_TREELSTM) a.hlr[b * H + ej] = e_h[0] + e_h[NC - 1];
    }
    w.advance();
  }
  tail_leave(w.gsync, a.plan.wgs);
}

// ------------------------------------------------------------------ backward
// The rows nobody sends a gradient to are the groups' first lists: elementwise, a barrier more for each group and a launch
// (4.8 us and the 4.5 in front of it) less.  16 chains of 20, H = 128: 2656 -> 2562 us (16 steps).
template <int MODEL, int GPW, bool WIDE>
__global__ __launch_bounds__(512, 1) void group_bwd_kernel(GroupBwdArgs a) {
  constexpr int NP = MODEL == GROUP_TREELSTM ? 3 : MODEL == GROUP_LSTM ? 1 : 2, NC = MODEL == GROUP_LSTM ? 1 : 2;
  // the product over a row of dA (K = 3H, 4H, H): k-groups of a wavefront, and float4 per lane and row
  constexpr int NL = MODEL == GROUP_TREELSTM ? 3 * GPW : MODEL == GROUP_LSTM ? 4 * GPW : GPW, Q = (NL + 3) / 4;
  constexpr int NG = MODEL == GROUP_TREELSTM ? 6 : MODEL == GROUP_LSTM ? 5 : 1;
  extern __shared__ __attribute__((aligned(16))) float red[];
  __shared__ int4 s_rec[2][2 * kGroupRows];
  __shared__ int s_bail;
  GroupWalk w;
  if (!w.start(a.plan, s_rec, &s_bail)) return;
  const int H = a.H, KG = H / 16, tid = threadIdx.x, lane = tid & 63, ks = tid >> 6;
  const int x = lane & 15, slot = lane >> 4, ej = w.ct * 16 + x;
  const int LG = MODEL == GROUP_TREELSTM ? 3 * KG : MODEL == GROUP_LSTM ? 4 * KG : KG;  // k-groups of dA's product

  // weights: wl for the product over dA (Tree-FC: for the left child), ws for the second kind (Tree-LSTM: U_f^T,
  // shared by both children; Tree-FC: the right child)
  constexpr int NS = MODEL == GROUP_LSTM ? 1 : GPW;
  float4 wl[NL], ws[NS];
  {
    const float4 *base = reinterpret_cast<const float4 *>(a.WTp) + slot * 16 + x;
    const long cols = MODEL == GROUP_TREEFC ? 2 * KG : KG;  // column tiles of the transposed matrix
#pragma unroll
    for (int i = 0; i < NL; i++) {
      const int kg = ks * NL + i;
      wl[i] = sel4(kg < LG, base[((kg < LG ? kg : 0) * cols + w.ct) * 64]);
    }
#pragma unroll
    for (int i = 0; i < NS; i++) {
      const int kg = ks * GPW + i;
      const long k = kg < KG ? kg : 0;
      if constexpr (MODEL == GROUP_TREELSTM) ws[i] = sel4(kg < KG, base[3L * H * H / 4 + (k * KG + w.ct) * 64]);
      else if constexpr (MODEL == GROUP_TREEFC) ws[i] = sel4(kg < KG, base[(k * cols + KG + w.ct) * 64]);
      else ws[i] = zero4();
    }
  }
  // (beside a long product on another stream these go first)
  if (ks < 4) __builtin_amdgcn_s_setprio(3);
  else __builtin_amdgcn_s_setprio(2);
  const int og = (lane >> 2) & 3;
  int kl[Q];  // this lane's float4 of a row of dA
  int in[Q];  // (a mask: as in the forward kernel)
#pragma unroll
  for (int q = 0; q < Q; q++) {
    in[q] = 4 * q + og < NL && ks * NL + 4 * q + og < LG ? -1 : 0;
    kl[q] = in[q] ? 16 * (ks * NL + 4 * q + og) + 4 * slot : 0;
    asm("" : "+v"(in[q]));
  }
  int in_f = og < GPW && ks * GPW + og < KG ? -1 : 0;
  const int kf = in_f ? 16 * (ks * GPW + og) + 4 * slot : 0;  // of a row of dF
  asm("" : "+v"(in_f));
  WideBwd<MODEL, GPW> wide(a, __builtin_amdgcn_readfirstlane(ks), lane, red);
  if constexpr (WIDE) wide.clear();
  bool begun = false;  // (as in the forward kernel)
  __syncthreads();

  for (int r = 0; r < w.nlists; r++) {
    const int4 *rt = s_rec[r & 1];
    // (rows without a parent: nothing to multiply, nothing sent to them)
    const bool alone = w.cur.w & 2;
    const int n = w.cur.y < kGroupRows ? w.cur.y : kGroupRows, T = alone ? 0 : (n + 3) >> 2, TW = WIDE && !alone ? wide_tiles(n) : 0;
    w.begin(a.plan, r);
    // the operands of the children's pointwise part: everything but d c of the parent was written before this launch (a wavefront
    // without rows reads the first one's, a missing child and the states of a leaf's children what is there)
    const int eb = 4 * ks + slot;
    const bool eon = eb < n;
    const int4 rec = rt[eon ? 2 * eb : 0];
    int kid[NC], kdr[NC];
    float pf[NC];
    struct Kid {
      float g[NG], dr, c[2];
    } kd[NC];
    kid[0] = rec.y;
    kdr[0] = rec.w;
    if constexpr (NC == 2) {
      kid[NC - 1] = rec.z;
      kdr[NC - 1] = rt[eon ? 2 * eb + 1 : 1].x;
    }
    const int parent = max(rec.x, 0);
    pf[0] = pf[NC - 1] = 0.f;
    if constexpr (MODEL == GROUP_TREELSTM) {
      pf[0] = row_at(a.gates, parent, 6 * H)[3 * H + ej];
      pf[NC - 1] = row_at(a.gates, parent, 6 * H)[4 * H + ej];
    } else if constexpr (MODEL == GROUP_LSTM) {
      pf[0] = row_at(a.gates, parent, 5 * H)[H + ej];
    }
#pragma unroll
    for (int s = 0; s < NC; s++) {
      Kid &q = kd[s];
      q.c[0] = q.c[1] = 0.f;
      const int v = max(kid[s], 0);
      q.dr = row_at(a.dret, max(kdr[s], 0), H)[ej];
      if constexpr (MODEL == GROUP_TREEFC) {
        q.g[0] = row_at(a.h, v, H)[ej];
      } else {
        const float *g = row_at(a.gates, v, NG * H) + ej;
        long to_c = v >= a.leaf_rows ? reinterpret_cast<const char *>(row_at(a.G, v, NC * 2 * H) + H + ej) - reinterpret_cast<const char *>(g) : 0;
        asm("" : "+v"(to_c));  // (or it is a branch, and waits with it)
        const float *c = reinterpret_cast<const float *>(reinterpret_cast<const char *>(g) + to_c);
#pragma unroll
        for (int t = 0; t < NG; t++) q.g[t] = g[(long)t * H];
#pragma unroll
        for (int t = 0; t < NC; t++) q.c[t] = c[t * (NG == 6 ? 2 * H : 0)];
      }
    }

    struct Opnd {
      float4 l[Q], f[2];
    };
    const float *at_l = nullptr, *at_f = nullptr;
    auto rows = [&](int t) {
      // (rows past the list's end stand for its first row; their results are not written)
      const int i = 4 * t + (lane & 3);
      const int row = rt[2 * (i < n ? i : 0)].x;
      at_l = row_at(a.dA, row, a.ld);
      if constexpr (MODEL == GROUP_TREELSTM) at_f = row_at(a.dF, row, 2 * H) + kf;
    };
    auto fetch = [&](Opnd &o) {
#pragma unroll
      for (int q = 0; q < Q; q++) o.l[q] = ld4(at_l + kl[q]);
      if constexpr (MODEL == GROUP_TREELSTM) {
        o.f[0] = ld4(at_f);
        o.f[1] = ld4(at_f + H);
      }
    };
    auto multiply = [&](int t, Opnd &o) {
#pragma unroll
      for (int q = 0; q < Q; q++) o.l[q] = and4(in[q], o.l[q]);
      if constexpr (MODEL == GROUP_TREELSTM) {
        o.f[0] = and4(in_f, o.f[0]);
        o.f[1] = and4(in_f, o.f[1]);
      }
      // (the long product in two accumulators: each MFMA would wait for the one before otherwise)
      floatx4 acc[NP], two = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int p = 0; p < NP; p++) acc[p] = floatx4{0.f, 0.f, 0.f, 0.f};
      unrolled<0, NL>([&](auto ic) {
        constexpr int i = decltype(ic)::value, q = i / 4, g = i % 4;
#pragma unroll
        for (int c = 0; c < 4; c++) {
          if constexpr (MODEL == GROUP_TREEFC) {
            acc[0] = mma4<g>(elem(o.l[q], c), elem(wl[i], c), acc[0]);
            acc[NP - 1] = mma4<g>(elem(o.l[q], c), elem(ws[i % NS], c), acc[NP - 1]);
          } else if (c & 1) {
            two = mma4<g>(elem(o.l[q], c), elem(wl[i], c), two);
          } else {
            acc[0] = mma4<g>(elem(o.l[q], c), elem(wl[i], c), acc[0]);
          }
        }
      });
      if constexpr (MODEL == GROUP_TREELSTM) {
        unrolled<0, GPW>([&](auto gc) {
          constexpr int g = decltype(gc)::value;
#pragma unroll
          for (int c = 0; c < 4; c++) {
            acc[1 % NP] = mma4<g>(elem(o.f[0], c), elem(ws[g], c), acc[1 % NP]);
            acc[2 % NP] = mma4<g>(elem(o.f[1], c), elem(ws[g], c), acc[2 % NP]);
          }
        });
      }
      if constexpr (MODEL != GROUP_TREEFC) {
#pragma unroll
        for (int k = 0; k < 4; k++) acc[0][k] += two[k];
      }
      SlotSums<NP> sums;
      sums.take(acc);
      sums.all();
      group_park<NP>(red, sums, t, ks, slot, x);
    };
    Opnd o, nx;
    const bool fours = 4 * TW < T;
    constexpr bool kEarly = !(WIDE && MODEL == GROUP_TREELSTM && GPW == 4);  // (its registers are full)
    if (kEarly && fours) rows(4 * TW);
    w.wait(a.plan, &s_bail);
    if constexpr (WIDE) {
      if (TW > 0 && !begun) wide.start(a, rt, n);
    }
    if (!kEarly && fours) rows(4 * TW);
    if (fours) fetch(o);
    float pdc = 0.f;
    if (MODEL != GROUP_TREEFC) pdc = ld_row((alone ? a.gates : row_at(a.dc, parent, H)) + ej);  // (never a row before its round: ld_row)
    if constexpr (WIDE)
      for (int t = 0; t < TW; t++) wide.tile(a, rt, n, t, t + 1 < TW, wl, ws, red);
    if (fours) {
      for (int t = 4 * TW; t + 1 < T; t++) {
        rows(t + 1);
        fetch(nx);
        multiply(t, o);
        o = nx;
      }
      multiply(T - 1, o);
    }
    arrived(MODEL != GROUP_TREEFC ? pdc : kd[NC - 1].g[0]);
    if (alone) pdc = pf[0] = pf[NC - 1] = 0.f;
    w.keep_next(r, s_rec);
    __syncthreads();
    if (s_bail) return;
    if constexpr (WIDE) {
      begun = r + 1 < w.nlists && w.nxt.z <= 0 && !(w.nxt.w & 2) && wide_tiles(w.nxt.y) > 0;
      if (begun) wide.start(a, s_rec[(r + 1) & 1], w.nxt.y < kGroupRows ? w.nxt.y : kGroupRows);
    }

    if (eon) {
      float v[NP];
#pragma unroll
      for (int p = 0; p < NP; p++) v[p] = 0.f;
      if (WIDE && ks < 4 * TW) wide_sum<NP>(red, ks, lane, v);
      else if (!alone) group_sum<NP>(red, ks, slot, x, v);
      int ee = ej;
      if (!kEarly) asm volatile("" : "+v"(ee));  // (or the rows' addresses are kept from list to list, in scratch memory)
#pragma unroll
      for (int s = 0; s < NC; s++) {
        const int c = kid[s];
        if (c < 0) continue;
        Kid &q = kd[s];
        if (c < a.leaf_rows) q.c[0] = q.c[1] = 0.f;
        float *d = row_at(a.dA, c, a.ld) + ee;
        if constexpr (MODEL == GROUP_TREELSTM) {
          const GateGrad gg = gate_grad(q.g[0], q.g[1 % NG], q.g[2 % NG], q.g[3 % NG], q.g[4 % NG], q.g[5 % NG], v[0] + v[(1 + s) % NP],
                                        pdc * pf[s], q.dr, q.c[0], q.c[1]);
          d[0] = gg.di; d[H] = gg.d_o; d[2 * H] = gg.du; d[3 * H] = gg.dfl + gg.dfr;
          if (c >= a.leaf_rows) {
            float *f = row_at(a.dF, c, 2 * H) + ee;
            f[0] = gg.dfl;
            f[H] = gg.dfr;
            row_at(a.dc, c, H)[ee] = gg.dc;
          }
        } else if constexpr (MODEL == GROUP_LSTM) {
          const LstmGateGrad gg = lstm_gate_grad(q.g[0], q.g[1 % NG], q.g[2 % NG], q.g[3 % NG], q.g[4 % NG], v[0], pdc * pf[0], q.dr, q.c[0]);
          d[0] = gg.di; d[H] = gg.df; d[2 * H] = gg.du; d[3 * H] = gg.d_o;
          if (c >= a.leaf_rows) row_at(a.dc, c, H)[ee] = gg.dc;
        } else {
          d[0] = treefc_dz(v[s % NP] + q.dr, q.g[0], a.act);
        }
      }
    }
    w.done();
    w.advance();
  }
  tail_leave(w.gsync, a.plan.wgs);
}

inline int group_lds(const void *kernel, size_t bytes) {
  CAVS_HIP_TRY(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
  return CAVS_OK;
}

template <class Args>
int group_launch(void (*kernel)(Args), size_t lds, const Args &a, void *stream) {
  const int H = a.H;
  const dim3 grid(8 * (H / 16) * ((a.plan.ngroups + 7) / 8));
  ResidentOrder order(as_stream(stream));
  if (order.rc()) return order.rc();
  launch(kernel, grid, 512, lds, as_stream(stream), a);
  CAVS_LAUNCH_CHECK();
  return CAVS_OK;
}

// One workgroup to a CU in any case; tiles of sixteen rows take what they need beyond that.
#define CAVS_GROUP_CASE(KERNEL, G, W, LDS)                                                    \
  {                                                                                           \
    constexpr size_t lds = (LDS) > kGroupLds ? (LDS) : kGroupLds;                             \
    static int attr = group_lds(reinterpret_cast<const void *>(KERNEL<MODEL, G, W>), lds);    \
    if (attr != CAVS_OK) return attr;                                                         \
    return group_launch(KERNEL<MODEL, G, W>, lds, a, stream);                                 \
  }
template <int MODEL, bool WIDE>
int group_fwd(const GroupFwdArgs &a, void *stream) {
  switch ((a.H + 127) / 128) {
    case 1: CAVS_GROUP_CASE(group_fwd_kernel, 1, WIDE, (WIDE ? WideFwd<MODEL, 1>::kLds : 0))
    case 2: CAVS_GROUP_CASE(group_fwd_kernel, 2, WIDE, (WIDE ? WideFwd<MODEL, 2>::kLds : 0))
    case 3: CAVS_GROUP_CASE(group_fwd_kernel, 3, WIDE, (WIDE ? WideFwd<MODEL, 3>::kLds : 0))
    default: CAVS_GROUP_CASE(group_fwd_kernel, 4, WIDE, (WIDE ? WideFwd<MODEL, 4>::kLds : 0))
  }
}
template <int MODEL, bool WIDE>
int group_bwd(const GroupBwdArgs &a, void *stream) {
  switch ((a.H + 127) / 128) {
    case 1: CAVS_GROUP_CASE(group_bwd_kernel, 1, WIDE, (WIDE ? WideBwd<MODEL, 1>::kLds : 0))
    case 2: CAVS_GROUP_CASE(group_bwd_kernel, 2, WIDE, (WIDE ? WideBwd<MODEL, 2>::kLds : 0))
    case 3: CAVS_GROUP_CASE(group_bwd_kernel, 3, WIDE, (WIDE ? WideBwd<MODEL, 3>::kLds : 0))
    default: CAVS_GROUP_CASE(group_bwd_kernel, 4, WIDE, (WIDE ? WideBwd<MODEL, 4>::kLds : 0))
  }
}
#undef CAVS_GROUP_CASE

// round_wide.hip has the kernels with tiles of sixteen rows
#define CAVS_GROUP_WIDE(M)                                                   \
  extern template int group_fwd<M, true>(const GroupFwdArgs &a, void *stream); \
  extern template int group_bwd<M, true>(const GroupBwdArgs &a, void *stream);
CAVS_GROUP_WIDE(GROUP_TREELSTM)
CAVS_GROUP_WIDE(GROUP_LSTM)
CAVS_GROUP_WIDE(GROUP_TREEFC)
#undef CAVS_GROUP_WIDE

}  // namespace cavs
