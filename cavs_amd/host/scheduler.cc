#include "scheduler.h"

#include <algorithm>
#include <cstring>

namespace cavs {

void Schedule::clear() {
  B = maxlen = N = executed = max_round = leaf_prefix = 0;
  batching = true;
  for (auto *v : {&sample_offset, &parent, &kids, &tids_to_jobids, &jobids_to_tids, &round2offset, &gather_ids[0], &gather_ids[1], &scatter_ids,
                  &root_tids, &bwd_rounds})
    v->clear();
  rounds.clear();
}

// LoadGraph, cavs/midend/graph_scheduler.cc:12-71.  Children in ascending vertex id (:52-58 appends in
// vertex order), two slots a vertex.
static std::string load_graph(const int32_t *g, int B, int maxlen, Schedule *s) {
  s->B = B;
  s->maxlen = maxlen;
  s->sample_offset.resize(B);
  int N = 0;
  for (int i = 0; i < B; i++) {
    const int32_t *row = g + (size_t)i * maxlen;
    int k = 0;
    while (k < maxlen && row[k] != -1) k++;
    if (k == maxlen) return "sample " + std::to_string(i) + " has no -1 terminator within maxlen";
    s->sample_offset[i] = N;
    N += k + 1;
  }
  s->N = N;
  s->parent.resize(N);
  s->kids.assign(2 * (size_t)N, -1);
  // (which of two slots a child takes, and below which child completes its parent, is as good as random:
  // both without a branch, 21 -> 8 ns per vertex for the schedule of 256 parse trees)
  std::vector<unsigned char> count(N, 0);
  int *parent = s->parent.data(), *kids = s->kids.data();
  unsigned crowded = 0;
  for (int i = 0; i < B; i++) {
    const int32_t *row = g + (size_t)i * maxlen;
    const int off = s->sample_offset[i], len = (i + 1 < B ? s->sample_offset[i + 1] : N) - off;
    for (int j = 0; j < len - 1; j++) {
      if (row[j] < 0 || row[j] >= len)
        return "sample " + std::to_string(i) + ": parent id out of range at vertex " + std::to_string(j);
      const int p = off + row[j];
      parent[off + j] = p;
      const unsigned n = count[p];
      count[p] = (unsigned char)(n < 2 ? n + 1 : 2);
      kids[2 * (size_t)p + (n != 0)] = off + j;
      crowded |= n & 2;
    }
    parent[off + len - 1] = -1;
  }
  for (int v = 0; crowded && v < N; v++) {
    const long n = count[v] < 2 ? 0 : std::count(s->parent.begin(), s->parent.end(), v);
    if (n > 2)
      return "vertex " + std::to_string(v) + " has " + std::to_string(n) + " children; the scheduler's gather lists hold two (graph_scheduler.h:16-18)";
  }
  return "";
}

static inline int nchild(const Schedule &s, int v) { return (s.kids[2 * (size_t)v] >= 0) + (s.kids[2 * (size_t)v + 1] >= 0); }

// BatchGraphScheduler::Initialize / ActivateNext, forward branch
// (cavs/midend/graph_scheduler.cc:169-193, 202-245).  One pass over the vertices in tensor-id order: a vertex
// joins the next round when the last of its children has its id.
static void batch_rounds(Schedule *s) {
  const int N = s->N;
  s->tids_to_jobids.assign(N + 1, 0);  // (one more: a candidate behind the last vertex)
  s->jobids_to_tids.assign(N, 0);
  s->scatter_ids.resize(N);
  for (auto &g : s->gather_ids) g.resize(N);
  s->round2offset.assign(1, 0);
  std::vector<int> waiting(N);  // children that have not run
  const int *parent = s->parent.data(), *kids = s->kids.data();
  int *job = s->tids_to_jobids.data(), *tid = s->jobids_to_tids.data(), *scatter = s->scatter_ids.data();
  int *gather[2] = {s->gather_ids[0].data(), s->gather_ids[1].data()}, gathers[2] = {0, 0}, scatters = 0;
  int begin = 0, end = 0;  // current round = tids [begin, end)
  for (int v = 0; v < N; v++) {
    const int n = (kids[2 * (size_t)v] >= 0) + (kids[2 * (size_t)v + 1] >= 0);
    waiting[v] = n;
    if (n == 0 && parent[v] >= 0) {
      job[end] = v;
      tid[v] = end++;
    }
  }
  s->leaf_prefix = end;
  while (end > begin) {
    // lists this round exposes: gather lists were appended while the round was being
    // formed (below); the scatter list holds the non-root jobs in job order
    Round r;
    r.offset = begin;
    r.n = end - begin;
    for (int c = 0; c < 2; c++) {
      r.gather_end[c] = gathers[c];
      r.gather_begin[c] = s->rounds.empty() ? r.gather_end[c] : s->rounds.back().gather_end[c];
    }
    r.scatter_begin = scatters;
    int next = end;
    for (int t = begin; t < end; t++) {
      const int p = parent[job[t]];
      if (p < 0) continue;
      scatter[scatters++] = t;
      job[next] = p;  // (stays if this was the last child; the next candidate overwrites it otherwise)
      tid[p] = next;
      next += --waiting[p] == 0;
    }
    for (int t = end; t < next; t++) {
      const int p = job[t];
      for (int i = 0; i < 2; i++) {
        const int c = kids[2 * (size_t)p + i];
        if (c >= 0) gather[i][gathers[i]++] = tid[c];
      }
      if (parent[p] < 0) s->root_tids.push_back(t);
    }
    r.scatter_end = scatters;
    s->rounds.push_back(r);
    s->max_round = std::max(s->max_round, r.n);
    s->round2offset.push_back(end);
    begin = end;
    end = next;
  }
  if (end < N) job[end] = 0;  // (a candidate that never became ready)
  s->tids_to_jobids.resize(N);
  s->scatter_ids.resize(scatters);
  for (int c = 0; c < 2; c++) s->gather_ids[c].resize(gathers[c]);
  s->executed = end;
  for (int k = (int)s->rounds.size() - 1; k >= 0; k--) s->bwd_rounds.push_back(k);
}

// SerialGraphScheduler (cavs/midend/graph_scheduler.cc:83-167): one vertex per round,
// tensor id == vertex id, samples one after the other, FIFO activation order.
static void serial_rounds(Schedule *s) {
  const int N = s->N;
  s->tids_to_jobids.assign(N, 0);
  s->jobids_to_tids.assign(N, 0);
  for (int v = 0; v < N; v++) s->tids_to_jobids[v] = s->jobids_to_tids[v] = v;
  std::vector<int> activated(N, 0), fifo;
  fifo.reserve(N);
  for (int i = 0; i < s->B; i++) {
    int lo = s->sample_offset[i], hi = i + 1 < s->B ? s->sample_offset[i + 1] : N;
    size_t head = fifo.size();
    for (int v = lo; v < hi; v++)
      if (nchild(*s, v) == 0 && s->parent[v] >= 0) fifo.push_back(v);
    for (; head < fifo.size(); head++) {
      int v = fifo[head], p = s->parent[v];
      if (p >= 0 && ++activated[p] == nchild(*s, p)) fifo.push_back(p);
    }
  }
  for (int v : fifo) {
    Round r;
    r.offset = v;
    r.n = 1;
    for (int c = 0; c < 2; c++) {
      r.gather_begin[c] = (int)s->gather_ids[c].size();
      if (nchild(*s, v) > c) s->gather_ids[c].push_back(s->kids[2 * (size_t)v + c]);
      r.gather_end[c] = (int)s->gather_ids[c].size();
    }
    r.scatter_begin = (int)s->scatter_ids.size();
    if (s->parent[v] >= 0) s->scatter_ids.push_back(v); else s->root_tids.push_back(v);
    r.scatter_end = (int)s->scatter_ids.size();
    s->rounds.push_back(r);
  }
  s->executed = (int)fifo.size();
  s->max_round = fifo.empty() ? 0 : 1;
  s->leaf_prefix = 0;
  // Backward order (ReverseGraph + the same FIFO, graph_scheduler.cc:73-81,110-140): roots
  // first, children after their parent.  The reference starts the next sample whenever
  // the vertex it pops has no forward children, i.e. at every leaf, not only at the end
  // of a sample; the order below reproduces that.
  std::vector<int> round_of(N, -1);
  for (size_t k = 0; k < s->rounds.size(); k++) round_of[s->rounds[k].offset] = (int)k;
  std::vector<int> bf;
  bf.reserve(N);
  auto init_sample = [&](int i) {
    int lo = s->sample_offset[i], hi = i + 1 < s->B ? s->sample_offset[i + 1] : N;
    for (int v = lo; v < hi; v++)
      if (s->parent[v] < 0 && nchild(*s, v) > 0) bf.push_back(v);
  };
  int sample_id = 0;
  init_sample(0);
  for (size_t head = 0; head < bf.size(); head++) {
    int v = bf[head];
    if (nchild(*s, v) > 0) {
      for (int k = 0; k < nchild(*s, v); k++) bf.push_back(s->kids[2 * (size_t)v + k]);
    } else if (++sample_id < s->B) {
      init_sample(sample_id);
    }
  }
  for (int v : bf) s->bwd_rounds.push_back(round_of[v]);
}

std::string build_schedule(const int32_t *graph, int B, int maxlen, bool batching, Schedule *out) {
  out->clear();
  out->batching = batching;
  if (!graph || B <= 0 || maxlen <= 0) return "empty graph feed";
  std::string err = load_graph(graph, B, maxlen, out);
  if (!err.empty()) return err;
  if (batching) batch_rounds(out); else serial_rounds(out);
  if (out->executed != out->N) {
    // A sample of a single vertex is never executed (graph_scheduler.cc:180); the schedule of the
    // rest stands, and it is the caller's business whether it accepts such a batch.  Any other
    // vertex that did not run sits on a parent cycle.
    int singles = 0;
    for (int i = 0; i < B; i++) {
      const int hi = i + 1 < B ? out->sample_offset[i + 1] : out->N;
      if (hi - out->sample_offset[i] == 1) singles++;
    }
    if (out->executed + singles != out->N)
      return std::to_string(out->N - out->executed - singles) + " vertices never become ready: the parent array holds a cycle "
             "(a vertex that is its own ancestor)";
  }
  return "";
}

std::string build_index_lists(const Schedule &s, int nch, int pairing, int *t2j, int *pair, int *child, int *roots) {
  const int N = s.N;
  std::copy(s.tids_to_jobids.begin(), s.tids_to_jobids.end(), t2j);
  if (s.executed != N) {  // (rows no round covers)
    std::fill(pair, pair + N, -1);
    std::fill(child, child + (size_t)nch * N, -1);
  }
  for (const Round &r : s.rounds) {
    const int m = r.scatter_end - r.scatter_begin;
    const int *sc = s.scatter_ids.data() + r.scatter_begin;
    if (pairing == 0) {
      std::copy(sc, sc + m, pair + r.offset);
      std::fill(pair + r.offset + m, pair + r.offset + r.n, -1);
    } else {
      std::fill(pair + r.offset, pair + r.offset + r.n, -1);
      for (int b = 0; b < m; b++) pair[sc[b]] = sc[b];
    }
    int *ch = child + (size_t)nch * r.offset;
    if (r.gather_begin[0] == r.gather_end[0] && r.gather_begin[1] == r.gather_end[1]) {  // a round of leaves
      std::fill(ch, ch + (size_t)nch * r.n, -1);
      continue;
    }
    for (int c = 0; c < nch; c++)
      if (r.gather_end[c] - r.gather_begin[c] != r.n)
        return "round at tensor id " + std::to_string(r.offset) + " mixes vertices with and without child " + std::to_string(c) +
               " (the reference's gather lists misalign there too)";
    const int *g0 = s.gather_ids[0].data() + r.gather_begin[0], *g1 = s.gather_ids[1].data() + r.gather_begin[1];
    if (nch == 1) {
      std::copy(g0, g0 + r.n, ch);
      if (r.gather_end[1] != r.gather_begin[1]) return "a chain vertex function got a vertex with two children";
    } else {
      for (int b = 0; b < r.n; b++) {
        ch[2 * (size_t)b] = g0[b];
        ch[2 * (size_t)b + 1] = g1[b];
      }
    }
  }
  // (a sample ends with its root, load_graph)
  for (int i = 0; i < s.B; i++) roots[i] = (i + 1 < s.B ? s.sample_offset[i + 1] : N) - 1;
  return "";
}

bool build_forest_lists(const Schedule &s, int nch, int fused_limit, const int *pair, const int *child, int *kid_rows,
                        int *orphans, int *n_orphans) {
  const int N = s.N;
  *n_orphans = 0;
  auto leaf_round = [](const Round &r) { return r.gather_begin[0] == r.gather_end[0] && r.gather_begin[1] == r.gather_end[1]; };
  if (!s.batching || s.rounds.empty() || !leaf_round(s.rounds[0]) || s.rounds[0].n != s.leaf_prefix) return false;
  for (size_t k = 1; k < s.rounds.size(); k++)
    if (leaf_round(s.rounds[k]) || s.rounds[k].n > fused_limit) return false;  // every round with children runs as a fused launch
  std::vector<int> writer(N, -1);  // of a pool row; -2: read
  for (int v = 0; v < N; v++) {
    const int p = pair[v];
    if (p < 0) {
      orphans[(*n_orphans)++] = v;
      continue;
    }
    if (p >= N || writer[p] >= 0) return false;  // two writers of one pool row
    writer[p] = v;
  }
  int unread = N - *n_orphans;
  for (const Round &r : s.rounds)
    for (size_t i = (size_t)nch * r.offset; i < (size_t)nch * (r.offset + r.n); i++) {
      kid_rows[i] = -1;
      const int p = child[i];
      if (p < 0) continue;
      // reads a row nobody wrote, or a second reader, or a reader in a round not after its writer's
      if (p >= N || writer[p] < 0 || writer[p] >= r.offset) return false;
      kid_rows[i] = writer[p];
      writer[p] = -2;
      unread--;
    }
  return unread == 0;  // (a message nobody reads: its gradient is whatever the pool holds)
}

// The trees of the message flow among the rows from `lo` on: comp[v] the tree of row v (v >= lo), weight its rows.
static void label_trees(const int *kid_rows, int nch, int N, int lo, std::vector<int> *comp_out, std::vector<int> *weight) {
  comp_out->assign((size_t)N + 1, -1);
  weight->clear();
  int *comp = comp_out->data();
  for (int v = N - 1; v >= lo; v--) {  // a row's consumer sits in a later round: parents come first
    if (comp[v] < 0) {
      comp[v] = (int)weight->size();
      weight->push_back(0);
    }
    (*weight)[comp[v]]++;
    // (rows before `lo` and missing children too: without a branch that is as good as random)
    for (int i = 0; i < nch; i++) {
      const int c = kid_rows[(size_t)nch * v + i];
      comp[c < 0 ? N : c] = comp[v];
    }
  }
}

// Which rounds run inside the tail launches, and who runs which row.  The rounds are a suffix of the
// forward order (a prefix of the backward order).  Inside it the message flow is a forest over slab
// rows (kid_rows: the rows whose messages a row consumes); a tree of that forest goes to one group
// as a whole, so nothing a group reads is written by another during the launch.  Trees are dealt
// heaviest first to the group with the fewest rows so far; the suffix starts at the earliest round
// from which no group gets more rows of a round than `lim`, nor more lists than `max_lists`.
void build_tail_lists(const Schedule &s, const int *kid_rows, int lim, int groups, int max_lists, int slice, TailLists *out,
                      int *rows_out) {
  *out = TailLists();
  const int R = (int)s.rounds.size(), N = s.N, G = groups, cap = max_lists;
  auto leaf_round = [](const Round &r) { return r.gather_begin[0] == r.gather_end[0] && r.gather_begin[1] == r.gather_end[1]; };
  if (lim <= 0 || G < 1 || G > 16 || slice < 1 || !s.batching || R < 3) return;
  int k0 = 1;
  while (k0 < R && (s.rounds[k0].n > G * lim || leaf_round(s.rounds[k0]))) k0++;
  std::vector<int> comp, weight, group, order, per;
  for (; R - k0 >= 2; k0++) {
    bool ok = true;
    for (int k = k0; k < R && ok; k++) ok = !leaf_round(s.rounds[k]);
    if (!ok) continue;
    const int lo = s.rounds[k0].offset;
    label_trees(kid_rows, 2, N, lo, &comp, &weight);
    order.resize(weight.size());
    for (size_t i = 0; i < order.size(); i++) order[i] = (int)i;
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return weight[a] > weight[b]; });
    group.assign(weight.size(), 0);
    int load[16] = {0};
    for (int c : order) {
      int best = 0;
      for (int g = 1; g < G; g++)
        if (load[g] < load[best]) best = g;
      group[c] = best;
      load[best] += weight[c];
    }
    // rows of round k that group g runs, and the lists that makes
    const int nr = R - k0;
    per.assign((size_t)G * nr, 0);
    for (int k = k0; k < R; k++)
      for (int b = s.rounds[k].offset; b < s.rounds[k].offset + s.rounds[k].n; b++) per[(size_t)group[comp[b]] * nr + (k - k0)]++;
    int lists = 0;
    for (int g = 0; g < G && ok; g++) {
      int mine = 0;
      for (int k = 0; k < nr; k++) {
        if (per[(size_t)g * nr + k] > lim) ok = false;
        mine += (per[(size_t)g * nr + k] + slice - 1) / slice;
      }
      if (mine > cap) ok = false;
      lists = std::max(lists, mine);
    }
    if (!ok) continue;
    TailLists &t = *out;
    t.first = k0;
    t.max_rounds = std::max(lists, 1);
    const size_t M = t.max_rounds;
    t.nrounds.assign(G, 0);
    for (auto *v : {&t.start, &t.count, &t.flags, &t.bstart, &t.bcount, &t.bflags}) v->assign((size_t)G * M, 0);
    // the device list: group by group, round by round
    std::vector<int> at((size_t)G * nr, -1);
    size_t fill = 0;
    for (int g = 0; g < G; g++)
      for (int k = 0; k < nr; k++) {
        at[(size_t)g * nr + k] = (int)fill;
        fill += per[(size_t)g * nr + k];
      }
    {
      std::vector<int> cur(at);
      for (int k = k0; k < R; k++)
        for (int b = s.rounds[k].offset; b < s.rounds[k].offset + s.rounds[k].n; b++) rows_out[cur[(size_t)group[comp[b]] * nr + (k - k0)]++] = b;
    }
    // A group's share of a round as lists of at most `slice` rows: the first waits for the rounds the
    // group has done so far, the last is an arrival.  Forward: rounds in order; backward: reversed.
    for (int g = 0; g < G; g++) {
      int tiles = 0;
      for (int dir = 0; dir < 2; dir++) {
        std::vector<int> &st = dir ? t.bstart : t.start, &ct = dir ? t.bcount : t.count, &fl = dir ? t.bflags : t.flags;
        int i = 0, done = 0;
        for (int kk = 0; kk < nr; kk++) {
          const int k = dir ? nr - 1 - kk : kk, c = per[(size_t)g * nr + k];
          for (int c0 = 0; c0 < c; c0 += slice, i++) {
            st[g * M + i] = at[(size_t)g * nr + k] + c0;
            ct[g * M + i] = std::min(slice, c - c0);
            fl[g * M + i] = ((c0 == 0 ? done : 0) << 1) | (c0 + slice >= c ? 1 : 0);
            if (!dir) tiles += (ct[g * M + i] + 3) / 4;
          }
          done += c > 0;
        }
        t.nrounds[g] = i;
      }
      t.tiles_max = std::max(t.tiles_max, tiles);
      t.lists_max = std::max(t.lists_max, t.nrounds[g]);
    }
    t.rows = fill;
    return;
  }
}

size_t group_lists_bound(const Schedule &s, size_t alone, int groups) {
  // records of the rows above the leaves forward and backward, and of the rows nobody sends a gradient to; lists of at least a
  // row each; two tables of groups
  const size_t inner = (size_t)(s.N - s.leaf_prefix);
  return inner * (16 + 8) + alone * (8 + 4) + 2 * (size_t)groups * 4;
}

// What the group with the most work spends on tiles when its lists run in tiles of four rows, and when they run in
// tiles of sixteen as far as they have more than eight rows.  In units of a tile of four rows, measured inside the
// launches at H = 512 (cycles): a tile of four 2580 forward and 2750 backward, of sixteen 6700 and 7000; the kernel with
// both kinds of tiles takes 0.15 longer over a list, so a batch whose lists are all short keeps the other one (chains of
// one row a group, H = 128: 2.88 against 3.02 ms per 16 steps; trees at H = 256, lists of 42, 27, 20 .. 1 rows: 2.57 against 2.39).
// The units are the Tree-LSTM's of that size; a tile's parts scale alike, and the choice is as good for the others: of 44 training sessions
// (chain LSTM and Tree-FC at H = 64 .. 512, Tree-LSTM at 64 .. 256, batches of 16 .. 256) it is the faster kind or within 1 %, where the
// two differ by up to 9 %.
static int group_tile_rows(const std::vector<int> &per, int rounds, int slice) {
  double four = 0, wide = 0;
  for (size_t i = 0; i < per.size(); i += rounds) {
    double f = 0, w = 0;
    for (int k = 0; k < rounds; k++)
      for (int c = per[i + k]; c > 0; c -= slice) {
        const int n = std::min(c, slice), w16 = (n + 7) / 16;
        f += (n + 3) / 4;
        w += 0.15 + 2.6 * w16 + (std::max(0, n - 16 * w16) + 3) / 4;
      }
    four = std::max(four, f);
    wide = std::max(wide, w);
  }
  return wide < four ? 16 : 4;
}

static constexpr int kUnevenShare = 64;

void build_group_lists(const Schedule &s, int nch, const int *t2j, const int *pair, const int *child, const int *kid_rows, const int *orphans,
                       int n_orphans, int lim, int groups, int slice, bool only_wide, int whole_from, GroupLists *out, int *block) {
  const bool back = orphans != nullptr;
  *out = GroupLists();
  const int R = (int)s.rounds.size(), N = s.N;
  auto leaf_round = [](const Round &r) { return r.gather_begin[0] == r.gather_end[0] && r.gather_begin[1] == r.gather_end[1]; };
  if (lim <= 0 || groups < 1 || slice < 1 || !s.batching || R < 3) return;
  int k0 = R;  // the rounds with children that no larger one follows (never that of the leaves: group_lists_bound)
  while (k0 > 1 && !leaf_round(s.rounds[k0 - 1]) && s.rounds[k0 - 1].n <= (long)groups * lim) k0--;
  std::vector<int> comp, weight, order, group, per, cell;
  for (; R - k0 >= 2; k0++) {
    const int lo = s.rounds[k0].offset, nr = R - k0;
    label_trees(kid_rows, nch, N, lo, &comp, &weight);
    // heaviest tree first to the group with the least so far
    const int G = std::min<int>(groups, (int)weight.size());
    order.resize(weight.size());
    for (size_t i = 0; i < order.size(); i++) order[i] = (int)i;
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return weight[a] > weight[b]; });
    group.assign(weight.size(), 0);
    std::vector<int> load(G, 0);
    for (int c : order) {
      const int best = (int)(std::min_element(load.begin(), load.end()) - load.begin());
      group[c] = best;
      load[best] += weight[c];
    }
    per.assign((size_t)G * nr, 0);
    bool ok = true;
    cell.resize(N - lo);  // which group's share of which round a row belongs to
    for (int k = k0; k < R; k++)
      for (int b = s.rounds[k].offset; b < s.rounds[k].offset + s.rounds[k].n; b++) {
        const int i = group[comp[b]] * nr + (k - k0);
        cell[b - lo] = i;
        ok &= ++per[i] <= lim;
      }
    // A share of more rows than a workgroup takes in two slices wants the groups evenly loaded: where few trees hold a round's
    // rows, most of the device would wait for one group.  Training steps of eight batches of few large trees, or of some among many small ones,
    // with shares of up to 512 however uneven / like this: Tree-LSTM H = 64 1.05 .. 1.65 times as long, 256 0.99 .. 1.41, 512 1.00 .. 1.24;
    // Tree-FC 0.98 (a tree of 1500 leaves among 255 of 10 .. 28) .. 1.48.
    for (int k = k0; k < R && ok && lim > kUnevenShare; k++)
      for (int g = 0; g < G && ok; g++) {
        const long share = per[(size_t)g * nr + (k - k0)];
        ok = share <= kUnevenShare || share * groups <= 2L * s.rounds[k].n;
      }
    if (!ok) continue;

    const int tile_rows = group_tile_rows(per, nr, slice);
    if (only_wide && tile_rows == 4) return;
    GroupLists &t = *out;
    t.first = k0;
    t.ngroups = G;
    t.rows = (size_t)(N - lo);
    t.tile_rows = tile_rows;
    // the records, group by group, round by round
    std::vector<int> at((size_t)G * nr), cur;
    int fill = 0;
    for (size_t i = 0; i < at.size(); i++) {
      at[i] = fill;
      fill += per[i];
    }
    // The rows whose message nobody reads open the backward pass: with the group whose tree they are in, those of earlier
    // rounds with any.
    std::vector<int> root_group(back ? n_orphans : 0), root_at((size_t)G + 1, 0);
    for (int i = 0, any = 0; i < (int)root_group.size(); i++) {
      const int b = orphans[i];
      root_group[i] = b >= lo ? group[comp[b]] : any++ % G;
      root_at[root_group[i] + 1]++;
    }
    for (int g = 0; g < G; g++) root_at[g + 1] += root_at[g];
    t.fwd.recs = 0;
    t.bwd.recs = t.rows * 8;
    // (word by word in place: as arrays that are copied, a record is stored in fours and loaded in sixteens, which the core
    // cannot forward -- 43 of 67 us for 4200 vertices)
    auto put = [](int *r, int a, int b, int c, int d, int e) {
      r[0] = a, r[1] = b, r[2] = c, r[3] = d, r[4] = e, r[5] = r[6] = r[7] = 0;
    };
    cur = at;
    int *const fwd = block + t.fwd.recs, *const bwd = block + t.bwd.recs;
    for (int b = lo; b < N; b++) {
      const size_t i = cur[cell[b - lo]]++;
      const int *c = child + (size_t)nch * b, *q = kid_rows + (size_t)nch * b;
      put(fwd + 8 * i, b, c[0], nch == 2 ? c[1] : -1, pair[b], t2j[b]);
      if (!back) continue;
      const int q0 = q[0], q1 = nch == 2 ? q[1] : -1;
      put(bwd + 8 * i, b, q0, q1, q0 >= 0 ? t2j[q0] : -1, q1 >= 0 ? t2j[q1] : -1);
    }
    cur.assign(root_at.begin(), root_at.end());
    for (size_t i = 0; i < root_group.size(); i++) {
      const int b = orphans[i];
      put(bwd + 8 * (t.rows + cur[root_group[i]]++), b, b, -1, t2j[b], -1);
    }
    size_t end = ((back ? 2 : 1) * t.rows + root_group.size()) * 8;
    // A direction: a group's share of a round as lists of at most `slice` rows; the first waits for the
    // rounds the group has done so far, the last is an arrival.
    for (int dir = 0; dir < (back ? 2 : 1); dir++) {
      GroupLists::Launch &l = dir ? t.bwd : t.fwd;
      l.groups = end;
      l.lists = end + (size_t)G * 4;
      int *lists = block + l.lists, nl = 0;
      for (int g = 0; g < G; g++) {
        int *gd = block + l.groups + 4 * (size_t)g, done = 0;
        gd[0] = nl;
        const int alone = dir ? root_at[g + 1] - root_at[g] : 0;
        for (int c0 = 0; c0 < alone; c0 += slice, nl++) {
          const int row[4] = {(int)t.rows + root_at[g] + c0, std::min(slice, alone - c0), 0, (c0 + slice >= alone) | 2};
          std::copy(row, row + 4, lists + 4 * (size_t)nl);
        }
        done += alone > 0;
        for (int i = 0; i < nr; i++) {
          const int k = dir ? nr - 1 - i : i, c = per[(size_t)g * nr + k], whole = !dir && s.rounds[k0 + k].n > whole_from ? 4 : 0;
          for (int c0 = 0; c0 < c; c0 += slice, nl++) {
            const int row[4] = {at[(size_t)g * nr + k] + c0, std::min(slice, c - c0), c0 == 0 ? done : 0, (c0 + slice >= c) | whole};
            std::copy(row, row + 4, lists + 4 * (size_t)nl);
          }
          done += c > 0;
        }
        gd[1] = nl - gd[0];
        gd[2] = done;
        gd[3] = 0;
      }
      end = l.lists + 4 * (size_t)nl;
    }
    t.ints = end;
    return;
  }
}

void schedule_from_lists(int B, int maxlen, int N, int nch, const int *round2offset, int R, const int *t2j,
                         const int *pair, const int *child, const int *roots, Schedule *out) {
  out->clear();
  Schedule &s = *out;
  s.B = B;
  s.maxlen = maxlen;
  s.N = N;
  s.batching = true;
  s.tids_to_jobids.assign(t2j, t2j + N);
  s.jobids_to_tids.assign(N, 0);
  for (int t = 0; t < N; t++) s.jobids_to_tids[t2j[t]] = t;
  s.round2offset.assign(round2offset, round2offset + R + 1);
  std::vector<char> is_root(N, 0);
  for (int i = 0; i < B; i++) is_root[roots[i]] = 1;
  // sample offsets and parents follow from the roots (each sample ends at its root) and the child lists
  s.sample_offset.assign(B, 0);
  for (int i = 1; i < B; i++) s.sample_offset[i] = roots[i - 1] + 1;
  s.parent.assign(N, -1);
  for (int r = 0; r < R; r++) {
    Round rd;
    rd.offset = round2offset[r];
    rd.n = round2offset[r + 1] - round2offset[r];
    for (int c = 0; c < 2; c++) rd.gather_begin[c] = (int)s.gather_ids[c].size();
    rd.scatter_begin = (int)s.scatter_ids.size();
    for (int b = 0; b < rd.n; b++) {
      const int t = rd.offset + b;
      for (int c = 0; c < nch; c++) {
        const int p = child[(size_t)nch * t + c];
        if (p < 0) continue;
        s.gather_ids[c].push_back(p);
        s.parent[t2j[p]] = t2j[t];
      }
      // the scatter list is the round's non-root jobs in job order under either pairing
      if (!is_root[t2j[t]]) s.scatter_ids.push_back(t); else s.root_tids.push_back(t);
    }
    for (int c = 0; c < 2; c++) rd.gather_end[c] = (int)s.gather_ids[c].size();
    rd.scatter_end = (int)s.scatter_ids.size();
    s.rounds.push_back(rd);
    s.max_round = std::max(s.max_round, rd.n);
  }
  (void)pair;
  s.executed = N;
  s.leaf_prefix = R > 0 ? round2offset[1] : 0;
  for (int k = R - 1; k >= 0; k--) s.bwd_rounds.push_back(k);
  s.kids.assign(2 * (size_t)N, -1);  // as load_graph builds them
  for (int v = 0; v < N; v++)
    if (s.parent[v] >= 0) {
      int *k = &s.kids[2 * (size_t)s.parent[v]];
      k[k[0] >= 0] = v;
    }
}

// trace_format: [N, R_fwd, R_bwd, then per round: offset, n_exec, exec..., n_g0, g0...,
// n_g1, g1..., n_s0, s0..., n_s1, s1..., n_init, init..., then tids_to_jobids (N),
// n_r2o, round2offset...].  Backward rounds are the forward rounds last to first with
// gather := recorded scatter lists and scatter := recorded gather lists
// (cavs/midend/graph_scheduler.cc:194-199, 246-257).
std::vector<int> Schedule::trace(bool with_backward) const {
  std::vector<int> o;
  auto put_list = [&](const int *p, int n) {
    o.push_back(n);
    o.insert(o.end(), p, p + n);
  };
  const int R = (int)rounds.size();
  o.push_back(N);
  o.push_back(R);
  o.push_back(with_backward ? (int)bwd_rounds.size() : 0);
  // forward gather_init list: the leaves of round 0 (batch) / the current leaf (serial)
  std::vector<int> init_fwd;
  if (batching && R) init_fwd.assign(tids_to_jobids.begin(), tids_to_jobids.begin() + rounds[0].n);
  for (int k = 0; k < R; k++) {
    const Round &r = rounds[k];
    o.push_back(r.offset);
    if (batching) put_list(&tids_to_jobids[r.offset], r.n); else put_list(&r.offset, 1);
    for (int c = 0; c < 2; c++) put_list(gather_ids[c].data() + r.gather_begin[c], r.gather_end[c] - r.gather_begin[c]);
    put_list(scatter_ids.data() + r.scatter_begin, r.scatter_end - r.scatter_begin);
    o.push_back(0);
    if (!batching && r.gather_end[0] == r.gather_begin[0]) init_fwd.assign(1, r.offset);
    put_list(init_fwd.data(), (int)init_fwd.size());
  }
  if (with_backward) {
    std::vector<int> init_bwd = batching ? root_tids : std::vector<int>();
    bool first = true;
    for (int k : bwd_rounds) {
      const Round &r = rounds[k];
      o.push_back(r.offset);
      if (batching) put_list(&tids_to_jobids[r.offset], r.n); else put_list(&r.offset, 1);
      if (batching) {
        put_list(scatter_ids.data() + r.scatter_begin, r.scatter_end - r.scatter_begin);
        o.push_back(0);
      } else {
        // serial backward: the gather list is one copy of the vertex per forward parent
        // (graph_scheduler.cc:158-161); the first round is set up by Initialize, which
        // fills no gather list (:100-107)
        int v = r.offset;
        int has_parent = parent[v] >= 0;
        if (first) o.push_back(0); else put_list(&v, has_parent);
        o.push_back(0);
        if (!has_parent) init_bwd.assign(1, v);
      }
      for (int c = 0; c < 2; c++) put_list(gather_ids[c].data() + r.gather_begin[c], r.gather_end[c] - r.gather_begin[c]);
      put_list(init_bwd.data(), (int)init_bwd.size());
      first = false;
    }
  }
  o.insert(o.end(), tids_to_jobids.begin(), tids_to_jobids.end());
  put_list(round2offset.data(), (int)round2offset.size());
  return o;
}

}  // namespace cavs
