"""Tiles of sixteen rows in the group launches (cavs_group_plan::tile_rows = 16) and of four at the list lengths where the kinds of
tiles change: every row against 64 bits, from the rows it read."""
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


def pre(A, W):
    """A W in 64 bits, and how far fp32 in any order may be off: K 2^-24 of the sum of the products' magnitudes (K additions and K roundings
    of products: twice that)"""
    A, W = A.astype(np.float64), W.astype(np.float64)
    return A @ W, 2.0 * W.shape[0] * 2.0 ** -24 * (np.abs(A) @ np.abs(W))


# exp and the reciprocal of the gates are good to 1e-7; a handful of operations behind them, on numbers of order one
GATE = 2.0 ** -20


def held(got, want, tol, what):
    got = got.astype(np.float64)
    assert np.isfinite(got).all(), what
    worst = (np.abs(got - want) - tol).max()
    assert worst <= 0, (what, worst, float(np.abs(got - want).max()), float(np.median(tol)))


def check_forward(model, H, res, W, xW, bias, rows, kid, pool0):
    """What a launch left for every row, from the children's rows it read (each row is written once)."""
    sig = lambda x: 1 / (1 + np.exp(-x))  # noqa: E731
    pool = res["pool"].reshape(len(pool0), -1)
    child = [np.where(kid[:, k, None] >= 0, pool[np.maximum(kid[:, k], 0)], np.float32(0)) for k in range(2)]
    h = [c[:, :H] for c in child]
    if model == "treefc":
        z, e = pre(np.concatenate(h, 1), W.reshape(2 * H, H))
        y = np.tanh(z + xW.reshape(-1, H)[rows] + bias[:H])
        for k in ("pool", "msg", "go"):
            held(res[k].reshape(len(pool0), -1)[rows], y, e + GATE, k)
        return
    c = [x[:, H:].astype(np.float64) for x in child]
    x4, b4 = xW.reshape(-1, 4, H)[rows].astype(np.float64), bias.reshape(4, H).astype(np.float64)
    if model == "lstm":
        z, e = pre(h[0], W.reshape(H, 4 * H))
        z, e = z.reshape(-1, 4, H) + x4 + b4, e.reshape(-1, 4, H)
        g = [sig(z[:, 0]), sig(z[:, 1]), np.tanh(z[:, 2]), sig(z[:, 3])]
        cc = g[0] * g[2] + g[1] * c[0]
        o, eo, ec = g[3], e[:, 3], e[:, 0] + e[:, 2] + e[:, 1] * np.abs(c[0])
    else:
        z, e = pre(h[0].astype(np.float64) + h[1], W[: 3 * H * H].reshape(H, 3 * H))
        z, e = z.reshape(-1, 3, H), e.reshape(-1, 3, H) + 2.0 ** -23 * (np.abs(h[0]) + np.abs(h[1])).sum(1)[:, None, None] * np.abs(W).max()
        f = [pre(h[k], W[3 * H * H:].reshape(H, H)) for k in range(2)]
        g = [sig(z[:, 0] + x4[:, 0] + b4[0]), sig(z[:, 1] + x4[:, 1] + b4[3]), np.tanh(z[:, 2] + x4[:, 2] + b4[2])]
        g += [sig(f[k][0] + x4[:, 3] + b4[1]) for k in range(2)]
        cc = g[0] * g[2] + g[3] * c[0] + g[4] * c[1]
        o, eo, ec = g[1], e[:, 1], e[:, 0] + e[:, 2] + f[0][1] * np.abs(c[0]) + f[1][1] * np.abs(c[1])
        held(res["hlr"][rows], h[0].astype(np.float64) + h[1], GATE * (1 + np.abs(h[0]) + np.abs(h[1])), "hlr")
    size = 1 + np.abs(c[0]) + np.abs(c[1])
    tc = np.tanh(cc)
    saved = res["gates"].reshape(len(pool0), -1, H)[rows]
    for k, v in enumerate(g + [tc]):
        held(saved[:, k], v, (e.max(1) if k < len(g) and model == "lstm" else ec + eo + e.max(1)) + GATE * size, f"gate {k}")
    for k in ("pool", "msg"):
        m = res[k].reshape(len(pool0), 2, H)[rows]
        held(m[:, 1], cc, ec + GATE * size, k + " c")
        held(m[:, 0], o * tc, ec + eo + GATE * size, k + " h")
    held(res["go"][rows], o * tc, ec + eo + GATE * size, "go")


def check_backward(model, H, res, W, base, lists, gates0, G0, dret, hpool, dc0):
    """What a launch left for every row that got a gradient, from its parent's row (none: alone)."""
    dA, gates = res["dA"].astype(np.float64), gates0.astype(np.float64)
    for recs, alone in lists:
        for side in range(1 if model == "lstm" else 2):
            v, k = recs[:, 0], recs[:, 1 + side]
            v, k = v[k >= 0], k[k >= 0]
            if not len(k):
                continue
            dr = dret.reshape(-1, H)[k].astype(np.float64)
            if model == "treefc":
                mh, e = pre(res["dA"].reshape(-1, H)[v], W.reshape(2 * H, H)[side * H: (side + 1) * H].T)
                mh, e = (0 * mh, 0 * e) if alone else (mh, e)
                y = hpool.reshape(-1, H)[k].astype(np.float64)
                held(res["dA"].reshape(-1, H)[k], (mh + dr) * (1 - y * y), e + GATE * (1 + np.abs(mh) + np.abs(dr)), f"dz {side}")
                continue
            if model == "lstm":
                mh, e = pre(res["dA"].reshape(-1, 4 * H)[v], W.reshape(H, 4 * H).T)
                pf = gates.reshape(-1, 5, H)[v, 1]
            else:
                mh, e = pre(res["dA"].reshape(-1, 4 * H)[v][:, : 3 * H], W[: 3 * H * H].reshape(H, 3 * H).T)
                m2, e2 = pre(res["dF"].reshape(-1, 2, H)[v, side], W[3 * H * H:].reshape(H, H).T)
                mh, e, pf = mh + m2, e + e2, gates.reshape(-1, 6, H)[v, 3 + side]
            mc = pf * res["dc"].reshape(-1, H)[v].astype(np.float64)
            if alone:
                mh, e, mc = 0 * mh, 0 * e, 0 * mc
            inner = (k >= base)[:, None]
            if model == "lstm":
                i, f, u, o, tc = gates.reshape(-1, 5, H)[k].transpose(1, 0, 2)
                cp = [np.where(inner, G0.reshape(-1, 2, H)[k, 1].astype(np.float64), 0.0)]
            else:
                i, o, u, fl, fr, tc = gates.reshape(-1, 6, H)[k].transpose(1, 0, 2)
                cp = [np.where(inner, G0.reshape(-1, 2, 2, H)[k, q, 1].astype(np.float64), 0.0) for q in range(2)]
            dh = mh + dr
            dc = mc + dh * o * (1 - tc * tc)
            size = (1 + np.abs(mh) + np.abs(dr) + np.abs(mc)) * (1 + sum(np.abs(x) for x in cp))
            # (gates0 are of (-1, 1): every factor behind d h is at most 1, x (1 - x) at most 2, and a c of an earlier row)
            tol = 4 * e * (1 + sum(np.abs(x) for x in cp)) + 8 * GATE * size
            want = [dc * u * i * (1 - i)]
            if model == "lstm":
                want += [dc * cp[0] * f * (1 - f), dc * i * (1 - u * u), dh * tc * o * (1 - o)]
            else:
                df = [dc * cp[0] * fl * (1 - fl), dc * cp[1] * fr * (1 - fr)]
                want += [dh * tc * o * (1 - o), dc * i * (1 - u * u), df[0] + df[1]]
            for q, x in enumerate(want):
                held(res["dA"].reshape(-1, 4, H)[k, q], x, tol, f"d gate {q} of child {side}")
            on = k >= base
            held(res["dc"][k][on], dc[on], tol[on], "dc")
            if model == "treelstm":
                for q in range(2):
                    held(res["dF"].reshape(-1, 2, H)[k, q][on], df[q][on], tol[on], "dF")


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
    # rows nobody sends a gradient to, each named as its own child, open the launch: slices of 32, the last of them an arrival
    alone = np.array([r for r in rows if r not in taken])
    arecs = np.full((len(alone), 8), -1, np.int32)
    arecs[:, 0] = arecs[:, 1] = arecs[:, 3] = alone
    _, blists = lists_of(tuple(reversed(sizes)))
    blists = [[N + c, min(32, len(alone) - c), 0, 2 | int(c + 32 >= len(alone))] for c in range(0, len(alone), 32)] + \
             [[at, n, wait + (wait > 0 or at == 0), flags] for at, n, wait, flags in blists]
    bgroups = [[0, len(blists), len(sizes) + 1, 0]]
    bdev = dict(groups=g.devi(bgroups), lists=g.devi(blists), recs=g.devi(np.concatenate([brecs[border], arecs])))
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
    for res in out.values():
        check_forward(model, H, res, W, xW, bias, rows, kid, pool0)
        check_backward(model, H, res, W, base, [(brecs, False), (arecs, True)], gates0, G0, dret, np.tanh(pool0), 0.1)
    assert (out[16]["pool"][base:] != pool0[base:]).any() and (out[16]["dA"] != dA0).any()
