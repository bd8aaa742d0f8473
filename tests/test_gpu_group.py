"""The launches that run many rounds at once at any hidden size of whole tiles up to 512
(cavs_*_group_fwd / _bwd): against the oracle, and against one launch per round."""
import ctypes as C

import numpy as np
import pytest

from cavs_amd import hip, session, synth
from test_gpu_models import compare, run_both
from test_oracle_models import small_workload
from tolerance import close

pytestmark = pytest.mark.gpu

MODELS = [("treelstm", "softmax", {}), ("lstm", "softmax", {}), ("treefc", "root_sq", dict(act=1, use_bias=True, use_x=True)),
          ("treefc", "root_sq", dict(act=0))]


@pytest.mark.parametrize("pairing", ["reference", "rowid"])
@pytest.mark.parametrize("H", [32, 96, 128, 160, 288])
@pytest.mark.parametrize("model,loss,kw", MODELS)
def test_rounds_of_every_hidden_size_against_the_oracle(oracle, model, loss, kw, H, pairing):
    w = small_workload(model, 411, B=45, H=H, E=12, V=31, C=5)
    if model == "treefc":  # (the spread the benchmark's weights have at their size: the tanh of a sum of 2H terms must not saturate)
        w["params"]["W"] *= np.float32(min(1.0, 0.25 * np.sqrt(64.0 / H)))
    compare(*run_both(oracle, w, loss=loss, pairing=pairing, **kw), loss)


@pytest.mark.parametrize("schedule,plan_cache,replay", [("host", 0, False), ("device", 0, False), ("host", 4, False), ("host", 4, True)])
@pytest.mark.parametrize("model,loss,kw", MODELS[:3])
def test_training_steps_with_and_without_the_launches(model, loss, kw, schedule, plan_cache, replay):
    """Three passes over two batches with the update in between (packed copies of the weights follow it),
    long chains among them (more lists than a group has rounds of 32 rows); host-built and
    device-built lists, cached plans, recorded graphs."""
    import torch

    H, E, V, C_ = 64, 12 if model == "treelstm" else 64, 31, 5
    ws = [small_workload(model, 500 + i, B=70, H=H, E=E, V=V, C=C_) for i in range(2)]
    if model == "lstm":
        for i, w in enumerate(ws):
            g, lens, rng = synth.chain_batch(77 + i, 70, 2, 90, 90)
            w.update(graph=g, N=sum(lens), x=np.floor(rng.bulk_uniform(sum(lens)) * V).astype(np.float32),
                     labels=np.floor(rng.bulk_uniform(sum(lens)) * C_).astype(np.float32))
    res = {}
    for tail in (-1, 0):
        s = session.Session(model, H=H, E=E, V=V, C_=C_, loss=loss, schedule=schedule, plan_cache=plan_cache, graph_replay=replay,
                            tail_rows=tail, **kw)
        p = {k: v for k, v in ws[0]["params"].items() if loss == "softmax" or not k.endswith("fc")}
        p["W"] = p["W"] * np.float32(0.25)
        s.set_params(p)
        feeds = [(w["graph"], torch.from_numpy(np.ascontiguousarray(w["x"], np.float32)).cuda(), torch.from_numpy(w["labels"]).cuda()) for w in ws]
        torch.cuda.synchronize()
        out = []
        for step in range(6):
            print(f"[case] {model} {schedule} cache={plan_cache} replay={replay} tail={tail} step {step}", flush=True)
            s.step(*feeds[step % 2], backward=True, lr=1e-2)
            out.append(dict(loss=s.fetch("loss"), go=s.fetch("graph_out"), **s.grads()))
        assert (s.counter("tail_rounds") > 0) == (tail == 0)
        res[tail] = out
        s.close()
    for a, b in zip(res[0], res[-1]):
        for k in b:
            close(a[k], b[k], k)


def test_a_wait_that_gives_up_leaves_the_launch():
    """One group, two lists, and one more arrival expected than there are workgroups: the bounded wait
    ends, the status word says so, every wave leaves."""
    import gpuutil as g

    hip.call("cavs_init", 0)
    H, N = 32, 3
    pool, xW, W, b = g.zeros(N, 2 * H), g.zeros(N, 4 * H), g.zeros(H, 4 * H), g.zeros(4 * H)
    G, gates, msg = g.zeros(N, 2 * H), g.zeros(N, 5 * H), g.zeros(N, 2 * H)
    groups = g.devi([[0, 2, 2, 0]])
    lists = g.devi([[0, 1, 0, 1], [1, 1, 1, 1]])
    recs = g.devi([[1, 0, -1, 1, 1, 0, 0, 0], [2, 1, -1, 2, 2, 0, 0, 0]])
    sync = g.devi(np.zeros(hip.lib().cavs_tail_sync_bytes() // 4))
    try:
        for extra, want in ((0, 0), (1, 1)):
            plan = hip.GroupPlan(g.P(groups), g.P(lists), g.P(recs), 1, g.P(sync), 64, extra)
            g.call("cavs_lstm_group_fwd", g.P(pool), g.P(xW), 4 * H, g.P(W), g.P(b), g.P(G), g.P(gates), g.P(msg), None, H, C.byref(plan),
                   g.stream())
            assert g.host(sync)[1] == want
        with pytest.raises(hip.CavsError):
            g.call("cavs_lstm_group_fwd", g.P(pool), g.P(xW), 4 * 48, g.P(W), g.P(b), g.P(G), g.P(gates), g.P(msg), None, 48, C.byref(plan),
                   g.stream())
    finally:
        g.release()


@pytest.mark.parametrize("H", [32, 96, 160, 288, 512])
@pytest.mark.parametrize("trees", [1, 20])
def test_an_infinity_reaches_what_multiplies_it_and_nothing_else(trees, H):
    """Tree-FC with relu, whose states have no bound.  Where some wavefronts have no column to multiply, or fewer than others, they read the
    first ones all the same: an infinite state of a leaf (forward) and an infinite gradient of a root (backward) come out as with a launch per
    round, in tiles of four rows (a tree a group) and of sixteen."""
    rng, B = np.random.default_rng(H), min(1900, trees * hip.lib().cavs_group_max_groups(H))
    graph = np.tile(np.array([2, 2, 4, 4, -1], np.int32), (B, 1))  # leaves 0, 1, 3, inner 2 = (0, 1), root 4 = (2, 3)
    params = dict(W=rng.uniform(-0.3, 0.3, (2 * H, H)).astype(np.float32), Bv=rng.uniform(0.1, 0.2, H).astype(np.float32))
    for at in (0, 4):
        x = rng.uniform(0.1, 0.5, (5 * B, H)).astype(np.float32)
        x[at, 0] = np.inf
        out = []
        for kw in ({}, dict(tail_rows=-1)):
            print(f"[case] H={H} B={B} infinite {'state' if at == 0 else 'gradient'} {kw}", flush=True)
            s = session.Session("treefc", H=H, E=0, V=0, C_=0, loss="root_sq", act=0, use_bias=True, use_x=True, **kw)
            s.set_params(params)
            s.step(graph, x, None, backward=True)
            assert (s.counter("tail_rounds") > 0) == (not kw)
            out.append([s.fetch("graph_out")] + list(s.grads().values()))
            s.close()
        go = out[0][0].reshape(B, 5, H)
        assert np.isfinite(go[1:]).all() and not np.isnan(go[0, 2]).any()
        if at == 0:
            assert (go[0, 2] == np.where(params["W"][0] > 0, np.inf, 0)).all()
        for a, b in zip(*out):
            np.testing.assert_array_equal(np.isnan(a), np.isnan(b))
            ok = np.isfinite(b)
            np.testing.assert_array_equal(np.isfinite(a), ok)
            close(np.where(ok, a, 0), np.where(ok, b, 0))
