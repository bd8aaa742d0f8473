"""What the barrier of the resident rounds (cavs_amd/csrc/round_sync.h) rests on, read off the machine code that
the kernels are compiled to.  Host only: no GPU."""
import os
import re
import subprocess

import pytest

from cavs_amd import build


def _assembly(name, tmp_path):
    out = str(tmp_path / (name + ".s"))
    cmd = [build.HIPCC] + [f for f in build.HIP_FLAGS if f != "-fPIC"] + ["-S", "--offload-device-only", os.path.join(build.CSRC, name), "-o", out]
    subprocess.run(cmd, check=True, capture_output=True)
    return [line.strip() for line in open(out) if re.match(r"\s+[a-z]", line) and not line.strip().startswith((".", ";"))]


@pytest.mark.parametrize("name,kernels", [("round_tail.hip", 3), ("round_group.hip", 24)])
def test_a_workgroup_leaves_behind_its_own_arrivals(tmp_path, name, kernels):
    """The last workgroup to leave zeroes the arrival words: every arrival must be acknowledged before the atomic
    that counts its workgroup as gone, or it could land on the zero and let the next launch's waits pass early."""
    code = _assembly(name, tmp_path)
    leaves = [i for i, line in enumerate(code) if line.startswith("global_atomic_add")]
    assert len(leaves) == kernels
    for i in leaves:
        for line in reversed(code[:i]):
            if re.match(r"s_waitcnt vmcnt\(0\)", line):
                break
            assert not re.match(r"(global|flat|buffer|scratch)_", line), f"{line!r} between the last complete wait and {code[i]!r}"
