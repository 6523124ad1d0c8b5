"""Raw workgroup barriers in the kernels (CPU, source text).

A loop that stages operands in LDS with a raw s_barrier lets other waves overwrite a buffer once the
barrier is passed, so the wait in front of it has to cover the wave's own LDS reads of that buffer
(lgkmcnt(0)) as well as its copies (vmcnt); the compiler adds neither to a raw barrier."""

import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "smolyax_amd", "csrc")


def test_raw_barriers_wait_for_lds_reads():
    seen = 0
    for path in sorted(glob.glob(os.path.join(CSRC, "*.hip"))):
        lines = open(path).read().split("\n")
        for i, line in enumerate(lines):
            if 'asm volatile("s_barrier"' not in line:
                continue
            seen += 1
            # the waits right before the barrier: every branch of them
            waits = []
            for k in range(i - 1, -1, -1):
                if "s_waitcnt" in lines[k]:
                    waits.append(lines[k])
                elif not re.search(r"^\s*(\}|else|if|issue|//)", lines[k]):
                    break
            assert waits, f"{path}:{i + 1}: no wait before the barrier"
            for w in waits:
                assert "vmcnt" in w and "lgkmcnt(0)" in w, f"{path}:{i + 1}: {w.strip()}"
    assert seen >= 4
