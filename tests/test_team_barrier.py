"""The team kernels' barrier on the instruction level: no member is counted in before the write-back
of its L2 has completed, and no wavefront leaves the barrier before the invalidation has."""
import os
import re
import subprocess

import pytest

from joltphysics_amd import build


def _team_assembly(tmp_path):
    try:
        cc = build.hipcc()
    except RuntimeError as e:
        pytest.skip(str(e))
    out = str(tmp_path / "team.s")
    subprocess.run([cc, *build.HIPCC_FLAGS, "-w", "-S", "--offload-device-only", "-x", "hip",
                    os.path.join(build.CSRC, "xpbd_team.hip"), "-I", os.path.join(build.ROOT, "include"), "-o", out],
                   check=True, capture_output=True)
    with open(out) as f:
        return [line.split(";")[0].strip() for line in f]


def test_cache_operations_are_waited_for(tmp_path):
    lines = _team_assembly(tmp_path)
    counts = {"buffer_wbl2": 0, "buffer_inv": 0}
    for k, line in enumerate(lines):
        name = line.split(" ")[0]
        if name not in counts:
            continue
        counts[name] += 1
        # up to the next access of global memory (the count, or a load behind the barrier), barrier or jump
        for after in lines[k + 1:]:
            if re.match(r"s_waitcnt .*vmcnt\(0\)", after):
                break
            assert not re.match(r"(flat|global|buffer|scratch)_|s_barrier|s_c?branch|s_endpgm", after), \
                f"line {k + 1}: {line} is not waited for before {after}"
    assert counts["buffer_wbl2"] > 0 and counts["buffer_inv"] > 0
