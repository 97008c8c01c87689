"""CPU: the host's choices of kernel (tests/cpp/dispatch_test.cpp answers with
the headers the runtime uses)."""
from __future__ import annotations

import subprocess

from conftest import PKG


def ask(lines):
    exe = PKG / "lib" / "dispatch_test"
    assert exe.exists(), "build with qora-llm-4b_amd/build.py"
    r = subprocess.run([str(exe)], input="\n".join(lines) + "\n", capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    out = r.stdout.splitlines()
    assert len(out) == len(lines)
    return out


def test_gqa_prefill_row_blocks_follow_the_cus():
    """32-row blocks up to 17.1875 tokens a CU, 4400 on 256; a device with an
    eighth of the CUs crosses at an eighth of the length; a forced packed
    order always has 48-row blocks."""
    ask_rows = lambda *q: [int(a) for a in ask([f"rows {s} {cus} {mode}" for s, cus, mode in q])]
    assert ask_rows((1, 256, 0), (4400, 256, 0), (4401, 256, 0), (4400, 256, 1), (300, 256, 2)) == [2, 2, 3, 2, 3]
    assert ask_rows((550, 32, 0), (551, 32, 0), (2200, 128, 0), (2201, 128, 0)) == [2, 3, 2, 3]
    assert ask_rows((2 ** 31 - 1, 256, 0), (2 ** 31 - 1, 1, 1)) == [3, 3]
