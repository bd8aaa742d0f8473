"""The production scheduler (cavs_amd/host/scheduler.cc) must expose bit-exactly the
rounds and index lists of the reference's schedulers.  Checked against the hand-derived
known answers and, over random batches, against the oracle.  Host only: no GPU."""
import functools
import json
import os

import numpy as np
import pytest

from cavs_amd import session, synth, hip

HERE = os.path.dirname(os.path.abspath(__file__))
KATS = json.load(open(os.path.join(HERE, "golden", "sched_kat.json")))["cases"]


@pytest.mark.parametrize("case", KATS, ids=[c["name"] for c in KATS])
def test_known_answers(case):
    tr = session.schedule_trace(np.array(case["graph"], np.int32))
    for k in ("N", "round2offset", "tids_to_jobids", "fwd", "bwd"):
        assert tr[k] == case[k], k


@functools.lru_cache(maxsize=None)
def _graphs():
    out = []
    for seed in range(10):
        out.append(synth.tree_batch(300 + seed, 1 + 3 * seed, 2, 5 + 6 * seed)[0])
    for seed in range(6):
        out.append(synth.chain_batch(400 + seed, 1 + 2 * seed, 2, 25)[0])
    out.append(synth.make_workload("C3")["graph"])
    out.append(synth.make_workload("C4")["graph"])
    return out


@pytest.mark.parametrize("idx", range(18))
@pytest.mark.parametrize("batching", [True, False])
def test_matches_oracle_bit_exact(oracle, idx, batching):
    graph = _graphs()[idx]
    want = oracle.sched_trace(graph, batching=batching)
    got = session.schedule_trace(graph, batching=batching)
    assert got["N"] == want["N"]
    assert got["tids_to_jobids"] == want["tids_to_jobids"]
    assert got["round2offset"] == want["round2offset"]
    assert len(got["fwd"]) == len(want["fwd"]) and len(got["bwd"]) == len(want["bwd"])
    for a, b in zip(got["fwd"] + got["bwd"], want["fwd"] + want["bwd"]):
        assert a == b


def test_rejects_malformed_feeds():
    with pytest.raises(hip.CavsError, match="terminator"):
        session.schedule_trace(np.array([[1, 2, 0]], np.int32))
    with pytest.raises(hip.CavsError, match="out of range"):
        session.schedule_trace(np.array([[5, -1, -1]], np.int32))
    with pytest.raises(hip.CavsError, match="3 children"):
        session.schedule_trace(np.array([[3, 3, 3, -1]], np.int32))
    with pytest.raises(hip.CavsError, match="single-vertex"):
        session.index_lists(np.array([[-1, -1], [1, -1]], np.int32), 1)
    with pytest.raises(hip.CavsError, match="cycle"):   # vertices 0 and 1 are each other's parent
        session.schedule_trace(np.array([[1, 0, 3, -1]], np.int32))
    with pytest.raises(hip.CavsError, match="cycle"):   # a vertex that is its own parent
        session.schedule_trace(np.array([[0, 2, -1]], np.int32))


@pytest.mark.parametrize("idx", range(18))
@pytest.mark.parametrize("pairing", ["reference", "rowid"])
def test_index_lists_match_the_oracles_schedule_and_invert(oracle, idx, pairing):
    """The lists the kernels consume (one entry per slab row) against the oracle's per-round
    lists, and back: the lists alone determine the complete schedule."""
    import arena

    graph = _graphs()[idx]
    tr = oracle.sched_trace(graph)
    nch = 2 if any(rd["gather"][1] for rd in tr["fwd"]) else 1
    want = arena.expected_arena(tr, graph, nch, pairing)
    got = session.index_lists(graph, nch, pairing)
    assert got["N"] == want["N"]
    for k in ("t2j", "pair", "child", "roots", "kid", "orphans"):
        assert got[k].tolist() == want[k].tolist(), k
    B, maxlen = graph.shape
    back = session.trace_from_lists(B, maxlen, nch, tr["round2offset"], got["t2j"], got["pair"], got["child"], got["roots"])
    assert back == session.schedule_trace(graph) == tr


def test_index_lists_refuse_mixed_arity_and_report_non_forests():
    with pytest.raises(hip.CavsError, match="mixes"):    # a chain inside a binary vertex function
        session.index_lists(np.array([[1, 2, -1]], np.int32), 2)
    with pytest.raises(hip.CavsError, match="two children"):
        session.index_lists(np.array([[2, 2, -1]], np.int32), 1)
    g = synth.tree_batch(7, 9, 2, 20)[0]
    assert session.index_lists(g, 2)["kid"] is not None
    assert session.index_lists(g, 2, fused_limit=3)["kid"] is None   # a round with children above the limit


def _check_tail_lists(graph, pairing, rows_limit, groups=8, max_lists=32):
    """Properties any deal must have, from the lists alone.  Returns the plan (or None)."""
    t = session.tail_lists(graph, pairing, rows_limit=rows_limit, groups=groups, max_lists=max_lists)
    lists = session.index_lists(graph, 2, pairing)
    tr = session.schedule_trace(graph)
    r2o = tr["round2offset"]
    if t is None:
        return None
    N, kid = lists["N"], lists["kid"].reshape(-1, 2)
    first, M = t["first"], t["M"]
    lo = r2o[first]
    round_of = np.searchsorted(np.asarray(r2o), np.arange(N), side="right") - 1
    owner = np.full(N, -1)
    # the slab rows from round `first` on, each exactly once
    assert sorted(t["rows"].tolist()) == list(range(lo, N))
    assert 1 <= first and len(r2o) - 1 - first >= 2
    for g in range(groups):
        n = int(t["nrounds"][g])
        assert 0 <= n <= M <= max_lists
        arrived, done_rounds, prev_round = 0, 0, -1
        for i in range(n):
            s, c, f = int(t["start"][g, i]), int(t["count"][g, i]), int(t["flags"][g, i])
            assert 1 <= c <= 32
            rows = t["rows"][s:s + c]
            rd = set(round_of[rows].tolist())
            assert len(rd) == 1, "a list holds rows of one round"
            k = rd.pop()
            assert k >= prev_round, "forward order"
            if k != prev_round:   # first slice of the group's share of this round: waits for all its earlier rounds
                assert f >> 1 == arrived, (g, i, f, arrived)
            else:                 # a further slice of the same round: no wait
                assert f >> 1 == 0
            prev_round = k
            owner[rows] = g
            last_slice = i + 1 == n or round_of[t["rows"][int(t["start"][g, i + 1])]] != k
            assert (f & 1) == int(last_slice), "a round's last slice is its arrival"
            arrived += f & 1
        # the backward lists: the same slices, rounds in reverse
        fwd = [(int(t["start"][g, i]), int(t["count"][g, i])) for i in range(n)]
        bwd = [(int(t["bstart"][g, i]), int(t["bcount"][g, i])) for i in range(n)]
        assert sorted(fwd) == sorted(bwd)
        brounds = [int(round_of[t["rows"][s]]) for s, _ in bwd]
        assert brounds == sorted(brounds, reverse=True)
        barrived = 0
        for i in range(n):
            f = int(t["bflags"][g, i])
            new_round = i == 0 or brounds[i] != brounds[i - 1]
            assert f >> 1 == (barrived if new_round else 0)
            barrived += f & 1
    assert (owner[lo:] >= 0).all()
    # no message crosses groups: a row's children inside the suffix belong to its group
    for v in range(lo, N):
        for c in kid[v]:
            if c >= lo:
                assert owner[c] == owner[v], (v, c)
    # no group gets more than the limit of any round
    for k in range(first, len(r2o) - 1):
        for g in range(groups):
            assert int(((round_of[lo:] == k) & (owner[lo:] == g)).sum()) <= rows_limit
    return t


@pytest.mark.parametrize("pairing", ["reference", "rowid"])
@pytest.mark.parametrize("seed,B,lmin,lmax", [(11, 64, 2, 56), (12, 24, 2, 56), (13, 200, 8, 40), (14, 7, 2, 9)])
def test_the_deal_of_trees_to_the_groups_of_the_tail_launches(seed, B, lmin, lmax, pairing):
    """Whole trees of the message flow per group, every row of the suffix exactly once, a group's share
    of a round in slices of at most 32 rows, wait / arrive flags that match the slices, the backward
    lists the forward ones reversed by round, and the limits kept."""
    graph = synth.tree_batch(seed, B, lmin, lmax, 2 * lmax - 1)[0]
    for limit in (4, 32, 96):
        t = _check_tail_lists(graph, pairing, limit)
        if B >= 24:
            assert t is not None, "a batch of this size has rounds to deal"
    _check_tail_lists(graph, pairing, 32, groups=3)


def test_the_deal_starts_later_under_a_tighter_limit_and_refuses_what_does_not_fit():
    graph = synth.tree_batch(21, 64, 2, 56, 111)[0]
    a, b = session.tail_lists(graph, rows_limit=32), session.tail_lists(graph, rows_limit=4)
    assert a["first"] < b["first"]
    assert len(a["rows"]) > len(b["rows"])
    # two lists per group cannot hold three rounds or more
    assert session.tail_lists(graph, rows_limit=32, max_lists=1) is None
    # a chain batch has no binary rounds to deal
    chain = synth.chain_batch(5, 6, 4, 9, 9)[0]
    with pytest.raises(hip.CavsError):
        session.tail_lists(chain)


@pytest.mark.parametrize("pairing", ["reference", "rowid"])
@pytest.mark.parametrize("nchild,B,lo,hi", [(2, 64, 2, 64), (2, 25, 2, 50), (2, 200, 8, 40), (1, 128, 10, 100), (1, 16, 20, 20)])
def test_the_lists_of_the_launches_that_keep_many_rounds_resident(nchild, B, lo, hi, pairing):
    """Every row above the leaves once per direction, with the neighbours the index lists give it; rows without a parent as the
    first lists of a backward pass, with the group their tree is in; a list waits for what its group has done."""
    graph = (synth.tree_batch if nchild == 2 else synth.chain_batch)(900 + B, B, lo, hi)[0]
    ix = session.index_lists(graph, nchild, pairing)
    N, kid = ix["N"], ix["kid"].reshape(-1, nchild)
    child = ix["child"].reshape(-1, nchild)
    g = session.group_lists(graph, nchild, pairing, rows_limit=64, groups=64)
    assert g["first"] >= 0
    lo_row = int(g["fwd"]["recs"][:, 0].min())
    none = np.full(N, -1)
    c1, k1 = (child[:, 1], kid[:, 1]) if nchild == 2 else (none, none)
    t2j = lambda k: np.where(k >= 0, ix["t2j"][np.maximum(k, 0)], -1)  # noqa: E731
    rows = N - lo_row
    f = g["fwd"]["recs"][:rows]
    v = f[:, 0]
    assert sorted(v) == list(range(lo_row, N))
    np.testing.assert_array_equal(f[:, 1:5], np.stack([child[v, 0], c1[v], ix["pair"][v], ix["t2j"][v]], 1))
    b = g["bwd"]["recs"][:rows]
    v = b[:, 0]
    assert sorted(v) == list(range(lo_row, N))
    np.testing.assert_array_equal(b[:, 1:5], np.stack([kid[v, 0], k1[v], t2j(kid[v, 0]), t2j(k1[v])], 1))
    alone = g["bwd"]["recs"][rows:]
    assert sorted(alone[:, 0]) == sorted(ix["orphans"])
    np.testing.assert_array_equal(alone[:, 1:5], np.stack([alone[:, 0], none[: len(alone)], ix["t2j"][alone[:, 0]], none[: len(alone)]], 1))
    for d in ("fwd", "bwd"):
        done_rows, seen = {}, np.zeros(len(g[d]["recs"]), int)
        for grp, (at, n, arrivals, _) in enumerate(g[d]["groups"]):
            arrived = 0
            for first, count, wait, flags in g[d]["lists"][at: at + n]:
                assert 1 <= count <= 32 and wait in (0, arrived)
                seen[first: first + count] += 1
                for r in g[d]["recs"][first: first + count]:
                    if d == "bwd" and flags & 2:
                        assert wait == 0 and not arrived
                        done_rows[int(r[0])] = (grp, -1)
                        continue
                    # who wrote what this row reads ran in an earlier, waited-for round of the same group
                    src = [int(k) for k in (kid[r[0]] if d == "fwd" else [])] or [int(r[0])]
                    for k in src:
                        if k >= lo_row and (k in done_rows or d == "fwd"):
                            assert done_rows[k][0] == grp and done_rows[k][1] < arrived
                    for k in ([int(r[0])] if d == "fwd" else [int(x) for x in kid[r[0]] if x >= 0]):
                        done_rows[k] = (grp, arrived)
                arrived += flags & 1
            assert arrived == arrivals
        assert (seen == 1).all()


@pytest.mark.parametrize("nchild,B,lo,hi", [(2, 64, 2, 64), (2, 25, 2, 50), (2, 256, 32, 256), (1, 128, 10, 100), (1, 16, 20, 20)])
def test_what_planning_a_new_batch_takes(nchild, B, lo, hi):
    """Room for the lists (pinned, and copied): by the rows that may be in them, not by all of the batch's.  Where the launches with tiles
    of four rows run instead, nothing of the block is written."""
    graph = (synth.tree_batch if nchild == 2 else synth.chain_batch)(900 + B, B, lo, hi)[0]
    N, leaves = session.index_lists(graph, nchild)["N"], int((session.index_lists(graph, nchild)["child"].reshape(-1, nchild)[:, 0] < 0).sum())
    g = session.group_lists(graph, nchild)
    assert g["room"] <= 24 * (N - leaves) + 12 * B + 8 * 64
    assert g["written"] <= g["room"]
    few = session.group_lists(graph, nchild, rows_limit=1 << 20, groups=64, only_wide=True)
    assert few["first"] < 0 or few["tile_rows"] == 16
    assert few["first"] >= 0 or few["written"] == 0
    assert session.group_lists(graph, nchild, rows_limit=1 << 20, groups=64)["first"] >= 0
    fwd = session.group_lists(graph, nchild, forward_only=True)
    assert fwd["first"] == g["first"] and fwd["bwd"] is None
    np.testing.assert_array_equal(fwd["fwd"]["recs"], g["fwd"]["recs"])


@pytest.mark.parametrize("large", [1, 3, 64])
def test_a_large_share_wants_the_groups_evenly_loaded(large):
    """Eight groups: a round is resident with more than 64 of its rows in one group only where that is at most twice an even share."""
    rng = synth.SplitMix64(51)
    trees = [synth.random_binary_tree(rng, 900 if i < large else 2) for i in range(64)]
    graph = synth.pack_graph(trees, 1799)
    sizes = np.diff(session.schedule_trace(graph)["round2offset"])
    for limit in (64, 512, 1 << 20):
        g = session.group_lists(graph, 2, rows_limit=limit, groups=8)
        share = np.zeros((8, len(sizes)), int)
        of = np.repeat(np.arange(len(sizes)), sizes)
        for i, (first, n, _, _) in enumerate(g["fwd"]["groups"]):
            for at, rows, _, _ in g["fwd"]["lists"][first:first + n]:
                np.add.at(share[i], of[g["fwd"]["recs"][at:at + rows, 0]], 1)
        most = share.max(0)
        assert (most <= limit).all() and ((most <= 64) | (8 * most <= 2 * sizes)).all()
        if large == 64 and limit == 1 << 20:
            assert most.max() > 512
