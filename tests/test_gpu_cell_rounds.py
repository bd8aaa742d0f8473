"""The rounds of a user's own vertex function in one launch per direction (the generated rounds_fwd / rounds_bwd)."""
import contextlib
import re
import subprocess

import numpy as np
import pytest

from cavs_amd import build
from test_cell_lowering import _declare, _dump
from test_gpu_cell import compare, run_generated
from test_gpu_resident import another_process
from test_oracle_models import small_workload


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
    got = []
    for turn in (contextlib.nullcontext, another_process):
        with turn():
            print(f"[case] {model} H={H} {'resident' if turn is contextlib.nullcontext else 'a launch per round'}", flush=True)
            got.append(run_generated(model, w, "reference", mode=1))
    assert got[0][3] == got[1][3] == 2
    compare(got[0], dict(loss=got[1][0], graph_out=got[1][1], grads=got[1][2]))

