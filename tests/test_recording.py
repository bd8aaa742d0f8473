"""What a session that records its steps asks of the device's runtime, and when: the host runtime over a stand-in for the
device (tests/native/device_standin.cc), in a process of its own.  Host only: no GPU."""
import os
import re
import subprocess
import sys

import pytest

from cavs_amd import build, hip

HERE = os.path.dirname(os.path.abspath(__file__))
DRIVER = """
import ctypes, sys
import numpy as np, torch
standin = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # in front of the backend in the order of symbols
standin.standin_faults.restype = ctypes.c_char_p
from cavs_amd import session, synth
def feeds(graph, C, H=0):  # feeds that count as the device's
    N = sum(int(np.argmax(row == -1)) + 1 for row in graph)
    return torch.zeros((N, H) if H else N), torch.zeros(N)
def chains(B, n):
    return synth.pack_graph([synth.chain(n)] * B, n)
def trees(B, leaves):
    rng = synth.SplitMix64(B)
    return synth.pack_graph([synth.random_binary_tree(rng, leaves) for _ in range(B)], 2 * leaves - 1)
%s
print(standin.standin_recorded(), standin.standin_replayed())
print(standin.standin_faults().decode(), end="")
"""


@pytest.fixture(scope="module")
def standin(tmp_path_factory):
    d = tmp_path_factory.mktemp("standin")
    src = os.path.join(HERE, "native", "device_standin.cc")
    own = set(re.findall(r"\b(cavs_[a-z0-9_]+)\(", open(src).read()))
    rest = d / "rest.c"  # every other entry point of the device: nothing is done
    rest.write_text("".join(f"int {n}() {{ return 0; }}\n" for n in sorted(set(hip._SIGS) - own)))
    subprocess.run(["gcc", "-fPIC", "-c", str(rest), "-o", str(d / "rest.o")], check=True, capture_output=True)
    subprocess.run([build.CXX] + build.CXX_FLAGS + ["-shared", src, str(d / "rest.o"), "-o", str(d / "standin.so")], check=True, capture_output=True)
    return str(d / "standin.so")


def run(standin, script):
    """(graphs recorded, launches of graphs, what the runtime was asked that it may not be)"""
    r = subprocess.run([sys.executable, "-c", DRIVER % script, standin], capture_output=True, text=True, timeout=300,
                       cwd=os.path.dirname(HERE))
    assert r.returncode == 0, r.stdout + r.stderr
    head, *faults = r.stdout.splitlines()
    return (*map(int, head.split()), faults)


def test_recorded_graphs_go_before_the_streams_they_ran_on(standin):
    """A session's graphs are given back before its streams, and none while a launch of it may be under way: not at the session's
    end, not where a fifth recording of a batch takes the place of the first."""
    recorded, replayed, faults = run(standin, """
s = session.Session("treefc", H=32, E=0, V=0, C_=5, loss="root_sq", plan_cache=2, graph_replay=True, use_x=True)
g = trees(4, 6)
xs = [feeds(g, 5, 32) for _ in range(6)]
s.step(g, *xs[0])
for x in xs:
    for _ in range(2):
        s.step(g, *x)
s.close()
""")
    assert recorded >= 5 and replayed > recorded
    assert faults == []


@pytest.mark.parametrize("model,loss,C,B,n", [("lstm", "softmax", 512, 300, 16), ("lstm", "softmax", 5, 20, 7), ("lstm", "softmax", 4096, 40, 9),
                                              ("treelstm", "softmax", 600, 300, 8), ("treelstm", "softmax", 5, 6, 9), ("treefc", "root_sq", 5, 6, 9),
                                              ("treefc", "sum_abs", 5, 20, 9), ("treelstm", "softmax", 5, 900, 7)])
def test_nothing_grows_while_a_step_is_recorded(standin, model, loss, C, B, n):
    """A batch seen forward only is trained on, and the other way round: what the passes need beyond that (sums of a wide
    head's gradients, chunk sums of biases, a workspace) is there before a pass is recorded, and both come to be recorded."""
    shape = "chains" if model == "lstm" else "trees"
    for first in (False, True):
        recorded, replayed, faults = run(standin, f"""
s = session.Session("{model}", H=64, E=64, V=50, C_={C}, loss="{loss}", plan_cache=2, graph_replay=True, use_x=True, use_bias=True)
g = {shape}({B}, {n})
x = feeds(g, {C}, {64 if model == "treefc" else 0})
for backward in ({first}, {not first}):
    for _ in range(5):
        s.step(g, *x, backward=backward, lr=0.1 if backward else 0.0)
s.close()
""")
        assert recorded >= 2 and replayed >= 5, (recorded, replayed)
        assert not [f for f in faults if "recorded" in f and "wait" in f]
