"""The rounds of a user's own vertex function in one launch per direction (the generated rounds_fwd / rounds_bwd)."""
import contextlib
import re
import subprocess

import numpy as np
import pytest

from cavs_amd import apps, build, session
from test_cell_lowering import _declare, _dump
from test_gpu_cell import NAMES, compare, run_generated
from test_gpu_resident import another_process
from test_oracle_models import small_workload
from tolerance import close


@pytest.mark.parametrize("model,H", [("treelstm2", 512), ("treegru", 100), ("treedeep", 64)])
def test_a_workgroup_leaves_behind_its_own_arrivals(model, H, tmp_path):
    """As for the hand-written launches: every arrival is acknowledged before the atomic that counts its workgroup as gone."""
    a = _declare(model, H)
    src, out = tmp_path / "rounds.hip", str(tmp_path / "rounds.s")
    src.write_text("#include <hip/hip_runtime.h>\n" + _dump(2))
    a.close()
    flags = [f for f in build.HIP_FLAGS if f != "-fPIC"]
    subprocess.run([build.HIPCC] + flags + ["-ffp-contract=off", "-S", "--offload-device-only", str(src), "-o", out], check=True, capture_output=True)
    text = open(out).read()
    assert "ScratchSize: 0" in text and not re.search(r"ScratchSize: [1-9]", text)
    code = [line.strip() for line in text.splitlines() if re.match(r"\s+[a-z]", line) and not line.strip().startswith((".", ";"))]
    leaves = [i for i, line in enumerate(code) if line.startswith("global_atomic_add")]
    assert len(leaves) == 2
    for i in leaves:
        for line in reversed(code[:i]):
            if re.match(r"s_waitcnt vmcnt\(0\)", line):
                break
            assert not re.match(r"(global|flat|buffer|scratch)_", line), line


def test_a_function_whose_weights_do_not_fit_keeps_a_launch_per_round():
    a = _declare("treelstm2", 544)
    assert _dump(2) == "" and _dump(1).startswith("#define")
    a.close()


@pytest.mark.gpu
@pytest.mark.parametrize("model", ["treelstm2", "treegate", "treegru", "treedeep"])
@pytest.mark.parametrize("H", [32, 100, 160, 288, 512])
def test_resident_rounds_give_what_a_launch_per_round_gives(model, H):
    """Sizes with one and with several k-groups a wavefront, one that is padded; lists of one row and of more than 32.  While another
    process has the GPU the same session runs a launch per round, which the oracle and fp64 autograd pin elsewhere; the two
    differ by the order of sums of at most 3H products."""
    # (weights whose spread shrinks with H: the gain of a level stays below one, so an early difference does not grow)
    w = small_workload(model, 187, B=60, H=H, E=12, V=29, C=5)
    for k in ("U", "W"):
        w["params"][k] = w["params"][k] * np.float32(0.4 * min(1.0, (64.0 / H) ** 0.5))
    got, counts = [], []
    for turn in (contextlib.nullcontext, another_process):
        with turn():
            print(f"[case] {model} H={H} {'resident' if turn is contextlib.nullcontext else 'a launch per round'}", flush=True)
            got.append(run_generated(model, w, "reference", mode=1, counts=counts))
    assert got[0][3] == got[1][3] == 2
    assert counts[0]["tail_rounds"] >= 2 * (counts[0]["rounds"] - 2) and counts[1]["tail_rounds"] == 0, counts
    compare(got[0], dict(loss=got[1][0], graph_out=got[1][1], grads=got[1][2]))


@pytest.mark.gpu
@pytest.mark.parametrize("model,H,mode", [("treelstm2", 100, 1), ("treedeep", 64, 1), ("treelstm", 64, 1), ("treelstm", 512, 1), ("lstm", 128, 1)])
@pytest.mark.parametrize("iters,read", [(1, False), (1, True), (3, False)])
def test_what_a_launch_that_gives_up_holds_back_is_run_again(model, H, mode, iters, read):
    """The waits of such a launch are bounded: when one runs out, the updates of that pass and of all behind it are held back.  A
    training loop that reads nothing, one that reads every step, one of three passes a Run: each ends where the same loop ends whose
    launches never give up (the rounds run as launches of their own from there on, so sums are ordered otherwise)."""
    batches = [small_workload(model, 500 + k, B=12, H=H, E=12, V=29, C=5) for k in range(5)]
    gain = np.float32(0.4 * min(1.0, (64.0 / H) ** 0.5))
    params = {k: np.asarray(batches[0]["params"][k], np.float32) * (gain if k in ("U", "W") else np.float32(1.0)) for k in NAMES[model]}
    maxlen = max(w["graph"].shape[1] for w in batches)
    graphs = [np.pad(w["graph"], ((0, 0), (0, maxlen - w["graph"].shape[1])), constant_values=-1) for w in batches]
    ends = []
    for gives_up in (False, True):
        w0 = batches[0]
        a = apps.App(model, B=12, maxlen=maxlen, H=H, E=w0["E"], V=w0["V"], C_=w0["C"], opt=session.OPT_BATCHING, lr=0.02, allow_fused=mode, iters=iters)
        a.set_params(params)
        seen = []
        for k, (g, w) in enumerate(zip(graphs, batches)):
            print(f"[case] {model} H={H} iters={iters} read={read} gives up={gives_up} step {k}", flush=True)
            if gives_up and k == 1:  # (64 polls, for one workgroup more than there are)
                a.bound_waits(64, 1)
            out = a.step(g, w["x"], w["labels"], train=True, fetch=read)
            if k == 0:
                assert a.counter("tail_rounds") > 0
            if read:
                seen.append(np.asarray(out[0]))
        values = {k: a.grad(k, np.shape(v), grad=False) for k, v in params.items()}
        grads = {k: a.grad(k, np.shape(v)) for k, v in params.items()}
        assert (a.counter("tail_rounds") > 0) == (not gives_up)
        a.close()
        ends.append((seen, values, grads))
    (seen, values, grads), (want_seen, want, want_grads) = ends[1], ends[0]
    for x, y in zip(seen, want_seen):
        close(x, y, "loss")
    for k in params:
        assert np.abs(want[k] - params[k].reshape(want[k].shape)).max() > 1e-4, f"{k} does not move"
        close(values[k], want[k], k)
        close(grads[k], want_grads[k], "d" + k)


def _trees_of_three_rounds(H, B=9):
    """Vertices of a sample: leaves 0, 1, 3, inner 2 = (0, 1), root 4 = (2, 3)"""
    graph = np.tile(np.array([2, 2, 4, 4, -1], np.int32), (B, 1))
    rng = np.random.default_rng(H)
    params = dict(W=rng.uniform(-0.3, 0.3, (2 * H, H)).astype(np.float32), Bv=rng.uniform(0.1, 0.2, H).astype(np.float32))
    x, mask = rng.uniform(0.1, 0.5, (5 * B, H)).astype(np.float32), np.zeros((5 * B, H), np.float32)
    mask[4::5] = 1
    return dict(graph=graph, x=x, labels=None, params=params, H=H, E=0, V=0, C=0, N=5 * B), mask


@pytest.mark.gpu
@pytest.mark.parametrize("H", [32, 64, 160, 288])
@pytest.mark.parametrize("where", ["state", "gradient"])
def test_an_infinity_reaches_what_multiplies_it_and_nothing_else(where, H):
    """Hidden sizes at which some wavefronts have no column to multiply, or fewer than others: an infinite state of one leaf (the first
    column, which such a wavefront reads all the same) makes its parent's row infinite or zero, an infinite gradient at one root
    an infinite gradient below, and neither a NaN -- as a launch per round has it."""
    w, mask = _trees_of_three_rounds(H)
    if where == "state":
        w["x"][0, 0] = np.inf
    else:
        mask[4, 0], w["x"][4, 0] = np.inf, 100.0  # (a column that relu passes)
    got, counts = [], []
    for turn in (contextlib.nullcontext, another_process):
        with turn():
            print(f"[case] infinite {where} H={H} {'resident' if turn is contextlib.nullcontext else 'a launch per round'}", flush=True)
            got.append(run_generated("treefc_xr", w, "rowid", mode=2, root_mask=mask, counts=counts))
    assert got[0][3] == got[1][3] == 2 and counts[0]["tail_rounds"] > 0 == counts[1]["tail_rounds"], counts
    go = got[0][1].reshape(-1, 5, H)
    assert not np.isnan(go[0, 2]).any() and np.isfinite(go[1:]).all()
    if where == "state":
        assert (go[0, 2] == np.where(w["params"]["W"][0] > 0, np.inf, 0)).all()
    else:
        assert not np.isnan(got[0][2]["dW"][:, 1:]).any() and np.isinf(got[0][2]["dW"][:, 1:]).any()
    for a, b in zip([got[0][1]] + list(got[0][2].values()), [got[1][1]] + list(got[1][2].values())):
        np.testing.assert_array_equal(np.isnan(a), np.isnan(b))
        close(np.where(np.isfinite(a), a, np.sign(np.nan_to_num(a, nan=0.0))), np.where(np.isfinite(b), b, np.sign(np.nan_to_num(b, nan=0.0))))
