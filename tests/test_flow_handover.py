"""The hand-over between workgroups of the dataflow launch
(gprat_amd/csrc/k_flow.hip), as compiled: a finished tile is written with
ordinary stores, so the L2 has to be written back, and the write-back has to
have ended, before the progress counter moves (a workgroup on another XCD
reads the tile as soon as it sees the counter). Whether that wait is there is
a matter of the compiled code: a release store's own wait was left out at one
of the hand-overs."""
import os
import re
import shutil
import subprocess

import pytest

from gprat_amd import build


def memory_operations(assembly):
    """(function, operations) of each function: its vector memory operations,
    barriers and waits for vector memory, in program order."""
    out, name = [], None
    for line in assembly.splitlines():
        m = re.match(r"(_Z\w+):", line)
        if m:
            name, ops = m.group(1), []
            out.append((name, ops))
        op = line.split(";")[0].strip()
        if name and re.match(r"(global|flat|scratch|buffer)_|s_barrier|s_waitcnt.*vmcnt\(0\)", op):
            ops.append(op)
    return out


def test_write_back_has_ended_before_the_counter_moves(tmp_path):
    if not (shutil.which(build.HIPCC) or os.path.exists(build.HIPCC)):
        pytest.skip("hipcc not available")
    asm = str(tmp_path / "k_flow.s")
    subprocess.run([build.HIPCC, *build.HIP_FLAGS, "--cuda-device-only", "-S", os.path.join(build.CSRC, "k_flow.hip"), "-o", asm],
                   check=True, capture_output=True)
    with open(asm) as f:
        functions = memory_operations(f.read())
    moved = 0
    for name, ops in functions:
        if "k_flow" not in name:
            continue
        for i, op in enumerate(ops):
            # only the counters are stored with agent scope
            if not re.match(r"global_store_dword .* sc1", op):
                continue
            moved += 1
            assert ops[i - 2] == "buffer_wbl2 sc1" and ops[i - 1].startswith("s_waitcnt"), (name, ops[i - 3:i + 1])
            # every wavefront's stores are in the L2 at the barrier before
            assert ops[i - 3] == "s_barrier" and ops[i - 4].startswith("s_waitcnt"), (name, ops[i - 6:i + 1])
    # factorisation: tiles, updates, both of the diagonal task's; solve: tiles, updates
    assert moved >= 6, [name for name, _ in functions]
