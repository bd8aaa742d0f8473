// The group launches (round_group.h): entry points, and the kernels with tiles of four rows.
#include "round_group.h"

namespace cavs {

static int group_plan(const char *who, const cavs_group_plan *p, int H, bool whole_lines, GroupPlan *out) {
  CAVS_REQUIRE(cavs_group_rounds_ok(H), "%s: H=%d (multiples of 32 up to %d)", who, H, kGroupMaxH);
  CAVS_REQUIRE(p && p->groups && p->lists && p->recs && p->sync, "%s: null plan", who);
  CAVS_REQUIRE(aligned16(p->groups) && aligned16(p->lists) && aligned16(p->recs), "%s: the plan must be 16-byte aligned", who);
  CAVS_REQUIRE(p->ngroups >= 1 && p->ngroups <= cavs_group_max_groups(H) && p->spin_max >= 0 && p->extra_arrivals >= 0,
               "%s: bad plan (1..%d groups)", who, cavs_group_max_groups(H));
  CAVS_REQUIRE(p->tile_rows == 0 || p->tile_rows == 4 || p->tile_rows == 16, "%s: tiles of %d rows (4 or 16)", who, p->tile_rows);
  *out = GroupPlan{reinterpret_cast<const int4 *>(p->groups), reinterpret_cast<const int4 *>(p->lists), reinterpret_cast<const int4 *>(p->recs),
                   p->sync, p->ngroups, H / 16, p->spin_max, std::min(H / 16 + p->extra_arrivals, 64), whole_lines, p->tile_rows == 16};
  return CAVS_OK;
}

static int treefc_group_fwd(const char *who, float *pool, const float *x, bool by_vertex, const float *Wp, const float *bias, float *G, float *msg,
                            float *graph_out, int H, int act, const cavs_group_plan *plan, void *stream) {
  GroupFwdArgs a{pool, x, H, Wp, bias, G, nullptr, nullptr, msg, graph_out, H, act, {}, by_vertex};
  if (int rc = group_plan(who, plan, H, line_rows(pool, H), &a.plan)) return rc;
  CAVS_REQUIRE(pool && Wp && G && msg && (act == 0 || act == 1), "%s: null pointer or act=%d", who, act);
  CAVS_REQUIRE(aligned16(pool) && aligned16(Wp), "%s: pool and Wp must be 16-byte aligned", who);
  return a.plan.wide ? group_fwd<GROUP_TREEFC, true>(a, stream) : group_fwd<GROUP_TREEFC, false>(a, stream);
}

}  // namespace cavs

using namespace cavs;

extern "C" {

int cavs_group_rounds_ok(int H) { return H > 0 && H % 32 == 0 && H <= kGroupMaxH ? 1 : 0; }
int cavs_group_max_groups(int H) { return cavs_group_rounds_ok(H) ? 8 * (kGroupWgsPerXcd / (H / 16)) : 0; }
int cavs_group_rows(void) { return kGroupRows; }

int cavs_treelstm_group_fwd(float *pool, const float *xW, int ld_xw, const float *Upk, const float *bias, float *G, float *hlr,
                            float *gates, float *msg, float *graph_out, int H, const cavs_group_plan *plan, void *stream) {
  GroupFwdArgs a{pool, xW, ld_xw, Upk, bias, G, hlr, gates, msg, graph_out, H, 0, {}};
  if (int rc = group_plan("cavs_treelstm_group_fwd", plan, H, line_rows(pool, 2 * H), &a.plan)) return rc;
  CAVS_REQUIRE(pool && xW && Upk && bias && G && hlr && gates && ld_xw >= 4 * H, "cavs_treelstm_group_fwd: null pointer or ld_xw=%d", ld_xw);
  CAVS_REQUIRE(aligned16(pool) && aligned16(Upk), "cavs_treelstm_group_fwd: pool and Upk must be 16-byte aligned");
  return a.plan.wide ? group_fwd<GROUP_TREELSTM, true>(a, stream) : group_fwd<GROUP_TREELSTM, false>(a, stream);
}

int cavs_lstm_group_fwd(float *pool, const float *xW, int ld_xw, const float *Whp, const float *bias, float *G, float *gates, float *msg,
                        float *graph_out, int H, const cavs_group_plan *plan, void *stream) {
  GroupFwdArgs a{pool, xW, ld_xw, Whp, bias, G, nullptr, gates, msg, graph_out, H, 0, {}};
  if (int rc = group_plan("cavs_lstm_group_fwd", plan, H, line_rows(pool, 2 * H), &a.plan)) return rc;
  CAVS_REQUIRE(pool && xW && Whp && bias && G && gates && ld_xw >= 4 * H, "cavs_lstm_group_fwd: null pointer or ld_xw=%d", ld_xw);
  CAVS_REQUIRE(aligned16(pool) && aligned16(Whp), "cavs_lstm_group_fwd: pool and Whp must be 16-byte aligned");
  return a.plan.wide ? group_fwd<GROUP_LSTM, true>(a, stream) : group_fwd<GROUP_LSTM, false>(a, stream);
}

int cavs_treefc_group_fwd(float *pool, const float *x, const float *Wp, const float *bias, float *G, float *msg, float *graph_out, int H,
                          int act, const cavs_group_plan *plan, void *stream) {
  return treefc_group_fwd("cavs_treefc_group_fwd", pool, x, false, Wp, bias, G, msg, graph_out, H, act, plan, stream);
}

int cavs_treefc_group_pull_fwd(float *pool, const float *x, const float *Wp, const float *bias, float *G, float *msg, float *graph_out, int H,
                               int act, const cavs_group_plan *plan, void *stream) {
  return treefc_group_fwd("cavs_treefc_group_pull_fwd", pool, x, true, Wp, bias, G, msg, graph_out, H, act, plan, stream);
}

int cavs_treelstm_group_bwd(float *dxW, int ld_dxw, float *dF, float *dc, const float *UTp, const float *gates, const float *G,
                            const float *dret, int leaf_rows, int H, const cavs_group_plan *plan, void *stream) {
  GroupBwdArgs a{dxW, ld_dxw, dF, dc, UTp, gates, G, nullptr, dret, H, leaf_rows, 0, {}};
  if (int rc = group_plan("cavs_treelstm_group_bwd", plan, H, line_rows(dxW, ld_dxw) && line_rows(dF, H) && line_rows(dc, H), &a.plan)) return rc;
  CAVS_REQUIRE(dxW && dF && dc && UTp && gates && G && dret && ld_dxw >= 4 * H && ld_dxw % 4 == 0 && leaf_rows >= 0,
               "cavs_treelstm_group_bwd: null pointer or ld=%d", ld_dxw);
  CAVS_REQUIRE(aligned16(dxW) && aligned16(dF) && aligned16(UTp), "cavs_treelstm_group_bwd: dxW, dF and UTp must be 16-byte aligned");
  return a.plan.wide ? group_bwd<GROUP_TREELSTM, true>(a, stream) : group_bwd<GROUP_TREELSTM, false>(a, stream);
}

int cavs_lstm_group_bwd(float *da, int ld_da, float *dc, const float *WhTp, const float *gates, const float *G, const float *dret,
                        int leaf_rows, int H, const cavs_group_plan *plan, void *stream) {
  GroupBwdArgs a{da, ld_da, nullptr, dc, WhTp, gates, G, nullptr, dret, H, leaf_rows, 0, {}};
  if (int rc = group_plan("cavs_lstm_group_bwd", plan, H, line_rows(da, ld_da) && line_rows(dc, H), &a.plan)) return rc;
  CAVS_REQUIRE(da && dc && WhTp && gates && G && dret && ld_da >= 4 * H && ld_da % 4 == 0 && leaf_rows >= 0,
               "cavs_lstm_group_bwd: null pointer or ld=%d", ld_da);
  CAVS_REQUIRE(aligned16(da) && aligned16(WhTp), "cavs_lstm_group_bwd: da and WhTp must be 16-byte aligned");
  return a.plan.wide ? group_bwd<GROUP_LSTM, true>(a, stream) : group_bwd<GROUP_LSTM, false>(a, stream);
}

int cavs_treefc_group_bwd(float *dz, const float *WTp, const float *h, const float *dret, int H, int act, const cavs_group_plan *plan,
                          void *stream) {
  GroupBwdArgs a{dz, H, nullptr, nullptr, WTp, nullptr, nullptr, h, dret, H, 0, act, {}};
  if (int rc = group_plan("cavs_treefc_group_bwd", plan, H, line_rows(dz, H), &a.plan)) return rc;
  CAVS_REQUIRE(dz && WTp && h && dret && (act == 0 || act == 1), "cavs_treefc_group_bwd: null pointer or act=%d", act);
  CAVS_REQUIRE(aligned16(dz) && aligned16(WTp), "cavs_treefc_group_bwd: dz and WTp must be 16-byte aligned");
  return a.plan.wide ? group_bwd<GROUP_TREEFC, true>(a, stream) : group_bwd<GROUP_TREEFC, false>(a, stream);
}

}  // extern "C"
