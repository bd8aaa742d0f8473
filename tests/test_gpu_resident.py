"""Launches that keep all their workgroups on the GPU: sessions of one process are put in order, processes that share
a GPU take turns."""
import contextlib
import ctypes as C
import fcntl
import subprocess
import sys
import threading

import numpy as np
import pytest

from cavs_amd import hip, session, synth
from test_oracle_models import small_workload
from tolerance import close

pytestmark = pytest.mark.gpu


@contextlib.contextmanager
def another_process():
    """Holds the lock as another process would: by a file description of its own."""
    hip.call("cavs_init", 0)
    bus = C.create_string_buffer(32)
    hip.call("cavs_device_bus_id", 0, bus, 32)
    with open(f"/sys/bus/pci/devices/{bus.value.decode().lower()}/vendor") as f:
        fcntl.flock(f, fcntl.LOCK_EX | fcntl.LOCK_NB)
        yield
        fcntl.flock(f, fcntl.LOCK_UN)


def _session(model, H, w, **kw):
    if model == "treefc":
        kw.update(loss="root_sq", act=1, use_bias=True, use_x=True)
    s = session.Session(model, H=H, E=12 if model == "treelstm" else H, V=31, C_=5, **kw)
    # (W from U(-0.4, 0.4) times this: a level of a Tree-FC tree multiplies the differences in its inputs by about
    # 0.4 / sqrt(3) times this times sqrt(2 H), 0.65 with the second form at every H, 1.3 at H = 256 with the first)
    spread = np.float32(0.25 * np.sqrt(64 / H) if model == "treefc" else 0.25)
    s.set_params({k: v * spread if k == "W" else v for k, v in w["params"].items() if model != "treefc" or not k.endswith("fc")})
    return s


@pytest.mark.parametrize("models", [(("treelstm", 512), ("lstm", 512)), (("treelstm", 512), ("treelstm", 512)), (("treefc", 256), ("lstm", 96))])
def test_sessions_on_threads_and_streams_of_their_own(models):
    """Two sessions train at a time, each on a thread and a stream of its own; every launch of either wants the whole
    GPU.  Each gives what it gives alone."""
    ws = [small_workload(m, 90 + i, B=60, H=H, E=12, V=31, C=5) for i, (m, H) in enumerate(models)]

    def train(i, out):
        (m, H), w = models[i], ws[i]
        s = _session(m, H, w)
        for k in range(30):
            s.step(w["graph"], w["x"], w["labels"], backward=True, lr=1e-4 if m == "treefc" else 1e-2)
            if k % 7 == i:
                s.sync()
        assert s.counter("tail_rounds") > 0
        out[i] = dict(loss=s.fetch("loss"), go=s.fetch("graph_out"), **s.grads())
        s.close()

    alone, together = [None, None], [None, None]
    for i in range(2):
        train(i, alone)
    threads = [threading.Thread(target=train, args=(i, together)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for a, b in zip(alone, together):
        for k in a:
            close(b[k], a[k], k)


@pytest.mark.parametrize("model,H,kw", [("treelstm", 512, {}), ("lstm", 128, {}), ("treefc", 256, dict(plan_cache=4, graph_replay=True)),
                                        ("treelstm", 96, dict(plan_cache=4)), ("treelstm", 64, dict(schedule="device"))])
def test_while_another_process_is_at_it_rounds_are_launches_of_their_own(model, H, kw):
    import torch

    w = small_workload(model, 12, B=50, H=H, E=12, V=31, C=5)
    feed = (w["graph"], torch.from_numpy(np.ascontiguousarray(w["x"], np.float32)).cuda(), torch.from_numpy(w["labels"]).cuda())
    torch.cuda.synchronize()
    s, plain = _session(model, H, w, **kw), _session(model, H, w, tail_rows=-1)
    free = contextlib.nullcontext
    # (the gradients of the sum of squares reach the tens: steps of 1e-2 would take W where the bound above no longer holds)
    lr = 1e-4 if model == "treefc" else 1e-2
    for k, turn in enumerate((another_process, another_process, free, free, free, another_process, free, free)):
        with turn():
            for one in (s, plain):
                one.step(*feed, backward=True, lr=lr)
            assert (s.counter("tail_rounds") > 0) == (turn is free), k
            for what in ("loss", "graph_out"):
                close(s.fetch(what), plain.fetch(what), what)
    for k, v in plain.grads().items():
        close(s.grads()[k], v, k)
    if "graph_replay" in kw:
        assert s.counter("graph_replays") > 0
    s.step(*feed, backward=True, lr=0.0)  # from here until somebody waits the lock is this process's
    with pytest.raises(BlockingIOError):
        with another_process():
            pass
    s.sync()
    with another_process():
        pass
    s.close()
    plain.close()


def test_a_session_made_while_another_process_is_at_it():
    """The device is asked once per process whether it runs such launches; a session made while that cannot be asked
    asks later.  In a process of its own, since this one has asked."""
    code = """
import sys
sys.path[:0] = sys.argv[1:]
from test_gpu_resident import another_process, _session, small_workload
w = small_workload("lstm", 12, B=50, H=64, E=12, V=31, C=5)
with another_process():
    s = _session("lstm", 64, w)
    s.step(w["graph"], w["x"], w["labels"], backward=True, lr=1e-2)
    s.sync()
    assert s.counter("tail_rounds") == 0 and s.counter("tail_ready") == 0
s.step(w["graph"], w["x"], w["labels"], backward=True, lr=1e-2)
s.sync()
assert s.counter("tail_rounds") > 0 and s.counter("tail_ready") == 1
print("done")
"""
    import os

    here = os.path.dirname(os.path.abspath(__file__))
    r = subprocess.run([sys.executable, "-c", code, os.path.dirname(here), here, os.path.join(os.path.dirname(here), "oracle")], capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.endswith("done\n"), r.stdout + r.stderr


@pytest.mark.parametrize("model,H,B", [("treelstm", 64, 40), ("treelstm", 64, 600), ("treelstm", 512, 600), ("lstm", 96, 1000), ("treefc", 64, 600)])
def test_a_forward_pass_plans_for_itself(model, H, B):
    """Without a backward pass only forward lists are made, in a large batch (4096 vertices) under the first product, and larger rounds by
    products leave the resident launch the others: what a launch per round gives (other orders of the same sums).  The backward pass
    that follows on the same batch has lists of its own."""
    w = small_workload(model, 77, B=B, H=H, E=12, V=31, C=5)
    assert (w["N"] >= 4096) == (B > 40)
    ref, s = (_session(model, H, w, tail_rows=k) for k in (-1, 0))
    few = _session(model, H, w, fused_round_rows=300)  # (rounds of more rows: products)
    for x in (ref, s, few):
        x.step(w["graph"], w["x"], w["labels"], backward=False)
    assert ref.counter("tail_rounds") == 0 and s.counter("tail_rounds") > 0 and few.counter("tail_rounds") > 0
    for x in (s, few):
        close(x.fetch("graph_out"), ref.fetch("graph_out"), "graph_out")
        close(x.fetch("loss"), ref.fetch("loss"), "loss")
    for x in (ref, s):
        x.step(w["graph"], w["x"], w["labels"], backward=True, lr=1e-3)
    got, want = s.grads(), ref.grads()
    for k, v in want.items():
        close(got[k], v, k)
    for x in (ref, s, few):
        x.close()


@pytest.mark.parametrize("H,B,resident", [(288, 1024, True), (288, 1040, False), (320, 1040, False), (352, 1040, True)])
def test_a_group_that_leaves_much_of_its_chiplet_idle_takes_128_rows(H, B, resident):
    """Chains of equal length in training: rounds of 128 rows a group (of eight) are resident at every size, rounds of 130 where a group
    is at least two thirds of its chiplet's workgroups; both ways what launches of their own give."""
    w = small_workload("lstm", 83, B=B, H=H, E=H, V=31, C=5, skew=False)
    s, ref = (_session("lstm", H, w, tail_rows=k) for k in (0, -1))
    for x in (s, ref):
        x.step(w["graph"], w["x"], w["labels"], backward=True, lr=1e-3)
    assert (s.counter("tail_rounds") > 0) == resident and ref.counter("tail_rounds") == 0
    close(s.fetch("graph_out"), ref.fetch("graph_out"), "graph_out")
    got, want = s.grads(), ref.grads()
    for name, v in want.items():
        close(got[name], v, name)
    for x in (s, ref):
        x.close()


@pytest.mark.parametrize("model,H,schedule,plan_cache", [("treelstm", 64, "host", 0), ("treelstm", 512, "device", 0), ("treefc", 96, "host", 2),
                                                         ("treefc", 256, "device", 2)])
def test_training_with_a_round_above_the_fused_limit(model, H, schedule, plan_cache):
    """A round of more rows than a fused launch is used for (2048) leaves a training pass's smaller rounds resident: what products
    and launches of their own give (other orders of the same sums), in both passes and on a batch seen before."""
    w = small_workload(model, 81, B=1700, H=H, E=12, V=31, C=5)
    sizes = np.diff(session.schedule_trace(w["graph"])["round2offset"])
    assert 2048 < sizes[1:].max() <= 4096
    # (a limit that is given is what it was)
    s, ref = _session(model, H, w, schedule=schedule, plan_cache=plan_cache), _session(model, H, w, fused_round_rows=2048)
    for k in range(2):
        for x in (s, ref):
            x.step(w["graph"], w["x"], w["labels"], backward=True, lr=1e-6)
        assert s.counter("tail_rounds") > 0 and ref.counter("tail_rounds") == 0
        close(s.fetch("graph_out"), ref.fetch("graph_out"), "graph_out")
        got, want = s.grads(), ref.grads()
        for name, v in want.items():
            close(got[name], v, name)
    for x in (s, ref):
        x.close()


@pytest.mark.parametrize("model,H,schedule,plan_cache", [("treelstm", 64, "host", 0), ("treelstm", 512, "device", 2), ("treefc", 64, "host", 2),
                                                         ("treefc", 256, "host", 0)])
def test_a_resident_round_above_the_fused_limit_keeps_relative_accuracy(model, H, schedule, plan_cache):
    """Pre-activations of 1e-6 .. 1e-3, and gates near 0 and 1, in a round of more than 2048 rows: relative errors of a few
    units, as the launches beside separate products give that ran such rounds.  Without weights, so that the pre-activations are what is declared."""
    w = small_workload(model, 81, B=1700, H=H, E=12, V=31, C=5)
    tr = session.schedule_trace(w["graph"])
    r2o, t2j = np.array(tr["round2offset"]), np.array(tr["tids_to_jobids"])
    big = int(np.argmax(np.diff(r2o)[1:])) + 1
    at = t2j[r2o[big]:r2o[big + 1]]
    assert 2048 < at.size <= 4096
    r = synth.SplitMix64(H)
    small = lambda n: (10.0 ** r.bulk_uniform(n, -6, -3) * np.where(r.bulk_uniform(n) < 0.5, -1, 1)).astype(np.float32)  # noqa: E731
    w["params"]["W"] = np.zeros_like(w["params"]["W"])
    if model == "treelstm":
        w["params"].update(U=np.zeros_like(w["params"]["U"]), Bv=np.concatenate([r.bulk_uniform(2 * H, -12, 6), small(H), r.bulk_uniform(H, -12, 6)]))
    else:
        w["params"]["Bv"] = np.zeros_like(w["params"]["Bv"])
        w["x"] = small(w["x"].size).reshape(-1, H)
    s = _session(model, H, w, schedule=schedule, plan_cache=plan_cache)
    for _ in range(2):
        s.step(w["graph"], w["x"], w["labels"], backward=True, lr=0.0)
        assert s.counter("tail_rounds") > 0
        got = s.fetch("graph_out")[at].astype(np.float64)
        if model == "treelstm":
            sig = lambda v: 1 / (1 + np.exp(-v.astype(np.float64)))  # noqa: E731
            bi, bf, bu, bo = np.asarray(w["params"]["Bv"], np.float32).reshape(4, H)
            c = s.fetch("msg_pool")  # (the children's states, as they are: their round may have the rounds' functions)
            child = np.array([[v for v in tr["fwd"][big]["gather"][k]] for k in (0, 1)])
            cl, cr = (c[child[k]][:, H:].astype(np.float64) for k in (0, 1))
            cc = sig(bi) * np.tanh(bu.astype(np.float64)) + sig(bf) * cl + sig(bf) * cr
            want = sig(bo) * np.tanh(cc)
        else:
            want = np.tanh(w["x"][at].astype(np.float64))
        # products of three gates, a sum of three terms of either sign: ten roundings of the terms' magnitudes
        mag = np.abs(want) if model == "treefc" else sig(bo) * (sig(bi) * np.abs(np.tanh(bu.astype(np.float64))) + sig(bf) * (np.abs(cl) + np.abs(cr)))
        assert (np.abs(got - want) <= 10 * 2.0 ** -23 * mag).all(), (np.abs(got - want) / mag).max()
    s.close()


@pytest.mark.parametrize("H,B,kw", [(32, 5, {}), (96, 40, {}), (256, 600, {}), (64, 600, dict(tail_rows=-1)), (64, 600, dict(fused_round_rows=300)),
                                    (40, 30, {})])
@pytest.mark.parametrize("shift", [0, 1])
def test_vertex_inputs_read_by_vertex(H, B, kw, shift):
    """Tree-FC: the leaves and the resident rounds read the caller's rows where they lie (also off a 16-byte boundary), rounds that are
    launches of their own have them brought into order: what rows in order give.  600 trees: more leaves than a fused launch's limit."""
    import torch

    w = small_workload("treefc", 91, B=B, H=H, E=12, V=31, C=5)
    s, ref = _session("treefc", H, w, **kw), _session("treefc", H, w, fused_round_rows=-1)
    room = torch.zeros(w["x"].size + 4, device="cuda")
    x = room[shift:shift + w["x"].size]
    x.copy_(torch.from_numpy(w["x"].reshape(-1)))
    for k in range(2):
        s.step(w["graph"], x.view(-1, H), torch.from_numpy(w["labels"]).cuda(), backward=True, lr=1e-6)
        ref.step(w["graph"], w["x"], w["labels"], backward=True, lr=1e-6)
        close(s.fetch("graph_out"), ref.fetch("graph_out"), "graph_out")
        got, want = s.grads(), ref.grads()
        for name, v in want.items():
            close(got[name], v, name)
    for z in (s, ref):
        z.close()


def test_a_wide_cell_leaves_middling_backward_rounds_to_products():
    """H = 1024, a batch with a round above the fused limit (1024): its backward rounds of more than 512 rows are products, what
    one launch of each gives (other orders of the same sums)."""
    w = small_workload("treelstm", 83, B=700, H=1024, E=12, V=31, C=5)
    sizes = np.diff(session.schedule_trace(w["graph"])["round2offset"])[1:]
    assert sizes.max() > 1024 and ((sizes > 512) & (sizes <= 1024)).any() and (sizes <= 512).any()
    s, ref = _session("treelstm", 1024, w), _session("treelstm", 1024, w, fused_round_rows=1024)
    for x in (s, ref):
        x.step(w["graph"], w["x"], w["labels"], backward=True, lr=1e-6)
    close(s.fetch("loss"), ref.fetch("loss"), "loss")
    got, want = s.grads(), ref.grads()
    for name, v in want.items():
        close(got[name], v, name)
    for x in (s, ref):
        x.close()
