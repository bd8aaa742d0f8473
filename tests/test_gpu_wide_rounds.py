"""Tiles of sixteen rows in the group launches (cavs_group_plan::tile_rows = 16) at the list lengths where the kinds of tiles
change, against the tiles of four rows, which the oracle pins elsewhere."""
import ctypes as C

import numpy as np
import pytest

from cavs_amd import hip, synth
from test_resident_barrier import test_a_workgroup_leaves_behind_its_own_arrivals as leaves_behind_its_own_arrivals


def test_a_workgroup_leaves_behind_its_own_arrivals(tmp_path):
    leaves_behind_its_own_arrivals(tmp_path, "round_wide.hip", 24)


def packed(W):
    """[K, cols] tile-major (CAVS_TASK_SGD_PACK): blocks of 16 k by 16 columns, a lane's four k together"""
    K, cols = W.shape
    return np.ascontiguousarray(W.reshape(K // 16, 4, 4, cols // 16, 16).transpose(0, 3, 1, 4, 2)).ravel()


def lists_of(sizes):
    """Lists of a group that runs its rounds in slices of 32 rows, and the groups table"""
    lists, at, done = [], 0, 0
    for n in sizes:
        for c in range(0, n, 32):
            lists.append([at + c, min(32, n - c), done if c == 0 else 0, int(c + 32 >= n)])
        at += n
        done += 1
    return [[0, len(lists), done, 0]], lists


def bound(K, a, b):
    """Two orders of a sum of K products of magnitudes a and b: each is within K 2^-24 of the sum of their magnitudes."""
    return 2.0 * K * 2.0 ** -24 * K * a * b


@pytest.mark.gpu
@pytest.mark.parametrize("H", [32, 96, 160, 256, 288, 512])
@pytest.mark.parametrize("model", ["treelstm", "lstm", "treefc"])
def test_sixteen_rows_a_tile_give_what_four_give(model, H):
    import gpuutil as g

    hip.call("cavs_init", 0)
    rng = synth.SplitMix64(900 + H)
    sizes = (70, 33, 32, 25, 24, 17, 16, 9, 8, 1)  # slices, whole tiles, the shortest rest worth a tile and the longest that is not
    N, base = sum(sizes), 40  # rows below `base` were written before the launch
    nc = 1 if model == "lstm" else 2
    ng, nw = {"treelstm": (6, 4), "lstm": (5, 4), "treefc": (0, 2)}[model]
    MW = H if model == "treefc" else 2 * H
    rows = base + np.arange(N)
    first = base + np.repeat(np.cumsum((0,) + sizes[:-1]), sizes)  # where the row's round begins
    kid = np.floor(rng.bulk_uniform(2 * N) * np.repeat(first, 2)).astype(np.int64).reshape(N, 2)
    kid[::11, 1] = -1  # a missing child
    if nc == 1:
        kid[:, 1] = -1
    W = (rng.bulk_normal(nw * H * H) / np.sqrt(H)).astype(np.float32)
    pool0 = (rng.bulk_normal((base + N) * MW).reshape(base + N, MW) * 0.5).astype(np.float32)
    xW = rng.bulk_normal((base + N) * (H if model == "treefc" else 4 * H)).astype(np.float32)
    bias = (rng.bulk_normal(4 * H) * 0.1).astype(np.float32)
    groups, lists = lists_of(sizes)
    recs = np.zeros((N, 8), np.int32)
    recs[:, 0], recs[:, 1:3], recs[:, 3], recs[:, 4] = rows, kid, rows, rows
    if model == "treelstm":
        wp = np.concatenate([packed(W[: 3 * H * H].reshape(H, 3 * H)), packed(W[3 * H * H:].reshape(H, H))])
        wt = np.concatenate([packed(np.ascontiguousarray(W[: 3 * H * H].reshape(H, 3 * H).T)), packed(np.ascontiguousarray(W[3 * H * H:].reshape(H, H).T))])
    else:
        M = W.reshape(H, 4 * H) if model == "lstm" else W.reshape(2 * H, H)
        wp, wt = packed(M), packed(np.ascontiguousarray(M.T))
    dev = dict(groups=g.devi(groups), lists=g.devi(lists), recs=g.devi(recs), wp=g.devf(wp), wt=g.devf(wt), xW=g.devf(xW), bias=g.devf(bias))
    # backward: rounds in reverse, every row the child of one row of an earlier list at most
    brecs = np.full((N, 8), -1, np.int32)
    taken = set()
    for i in range(N):
        brecs[i, 0] = rows[i]
        kids = []
        for k in kid[i][:nc]:
            kids.append(int(k) if k >= 0 and int(k) not in taken else -1)
            taken.add(int(k))
        kids += [-1] * (2 - len(kids))
        brecs[i, 1:3] = kids
        brecs[i, 3], brecs[i, 4] = max(kids[0], -1), max(kids[1], -1)
    border = np.concatenate([np.arange(sum(sizes[:r]), sum(sizes[: r + 1])) for r in reversed(range(len(sizes)))])
    bgroups, blists = lists_of(tuple(reversed(sizes)))
    bdev = dict(groups=g.devi(bgroups), lists=g.devi(blists), recs=g.devi(brecs[border]))
    gates0 = np.tanh(rng.bulk_normal(max(1, (base + N) * ng * H))).astype(np.float32)
    G0 = (rng.bulk_normal(nc * (base + N) * MW) * 0.5).astype(np.float32)
    dret = rng.bulk_normal((base + N) * H).astype(np.float32)
    ld = {"treelstm": 4 * H, "lstm": 4 * H, "treefc": H}[model]
    dA0 = (rng.bulk_normal((base + N) * ld) * 0.1).astype(np.float32)
    dF0 = (rng.bulk_normal(2 * (base + N) * H) * 0.1).astype(np.float32)
    out = {}
    try:
        for tile_rows in (4, 16):
            print(f"[case] {model} H={H} tiles of {tile_rows} rows", flush=True)
            sync = g.devi(np.zeros(hip.lib().cavs_tail_sync_bytes() // 4))
            pool, G, hlr = g.devf(pool0), g.zeros(nc * (base + N), MW), g.zeros(base + N, H)
            gates, msg, go = g.zeros(base + N, max(1, ng) * H), g.zeros(base + N, MW), g.zeros(base + N, H)
            plan = C.byref(hip.GroupPlan(g.P(dev["groups"]), g.P(dev["lists"]), g.P(dev["recs"]), 1, g.P(sync), 1 << 19, 0, tile_rows))
            if model == "treelstm":
                g.call("cavs_treelstm_group_fwd", g.P(pool), g.P(dev["xW"]), 4 * H, g.P(dev["wp"]), g.P(dev["bias"]), g.P(G), g.P(hlr), g.P(gates),
                       g.P(msg), g.P(go), H, plan, g.stream())
            elif model == "lstm":
                g.call("cavs_lstm_group_fwd", g.P(pool), g.P(dev["xW"]), 4 * H, g.P(dev["wp"]), g.P(dev["bias"]), g.P(G), g.P(gates), g.P(msg), g.P(go), H,
                       plan, g.stream())
            else:
                g.call("cavs_treefc_group_fwd", g.P(pool), g.P(dev["xW"]), g.P(dev["wp"]), g.P(dev["bias"]), g.P(G), g.P(msg), g.P(go), H, 1, plan, g.stream())
            assert not g.host(sync).any()
            res = dict(pool=g.host(pool), G=g.host(G), hlr=g.host(hlr), gates=g.host(gates), msg=g.host(msg), go=g.host(go))
            dA, dF, dc = g.devf(dA0), g.devf(dF0), g.zeros(base + N, H, fill=0.1)
            plan = C.byref(hip.GroupPlan(g.P(bdev["groups"]), g.P(bdev["lists"]), g.P(bdev["recs"]), 1, g.P(sync), 1 << 19, 0, tile_rows))
            if model == "treelstm":
                g.call("cavs_treelstm_group_bwd", g.P(dA), 4 * H, g.P(dF), g.P(dc), g.P(dev["wt"]), g.P(g.devf(gates0)), g.P(g.devf(G0)), g.P(g.devf(dret)),
                       base, H, plan, g.stream())
            elif model == "lstm":
                g.call("cavs_lstm_group_bwd", g.P(dA), 4 * H, g.P(dc), g.P(dev["wt"]), g.P(g.devf(gates0)), g.P(g.devf(G0)), g.P(g.devf(dret)), base, H,
                       plan, g.stream())
            else:
                g.call("cavs_treefc_group_bwd", g.P(dA), g.P(dev["wt"]), g.P(g.devf(np.tanh(pool0))), g.P(g.devf(dret)), H, 1, plan, g.stream())
            assert not g.host(sync).any()
            res.update(dA=g.host(dA), dF=g.host(dF), dc=g.host(dc))
            out[tile_rows] = res
    finally:
        g.release()
    # A pre-activation is a sum of at most 2H products of states (below 3) and weights (below 5 / sqrt(H)), a gradient one of 5H products of
    # gradients; ten rounds pass a difference on with a gain of order one.  The bound is far above what is seen.
    for k, want in out[4].items():
        scale = max(1.0, float(np.abs(want).max()))
        tol = 10 * bound(5 * H, 1.0, 1.0 / H) * scale
        assert np.isfinite(want).all() and np.abs(out[16][k].astype(np.float64) - want).max() <= tol, (k, np.abs(out[16][k] - want).max(), tol)
    assert (out[16]["pool"][base:] != pool0[base:]).any() and (out[16]["dA"] != dA0).any()
