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


def _tile_cases():
    """(tile named, gate/up, operand type, m, k, n) of the GPU tests."""
    import test_q4_gpu as t
    for name, m, k, n in t.GEMM_TILES:
        tile = name.replace("gate/up ", "").split()[0]
        for x_dtype in ("bf16",) if "bf16 x" in name else ("f16", "bf16"):
            yield tile, name.startswith("gate/up"), x_dtype, m, k, n
    for name, x_dtype, m, k, n in t.GEMM_TILES_BY_TYPE:
        yield name.replace("gate/up ", ""), name.startswith("gate/up"), x_dtype, m, k, n


def test_q4_gemm_sizes_take_the_tiles_they_name():
    cases = list(_tile_cases())
    got = ask([f"tile {m} {k} {n} {int(x == 'bf16')} {int(gu)} 256" for _, gu, x, m, k, n in cases])
    assert [(c, g) for c, g in zip(cases, got) if c[0] != g] == []


def test_q4_gemm_every_built_tile_is_tested():
    """Every tile of the table, form and operand type, in both device layouts
    (8- and 16-column tiles); no size takes the four left out (a wide search
    over m, k and n at 256 CUs)."""
    built = [b.split() for b in ask([f"built {t}" for t in range(64)]) if b != "-"]
    want = {(name, gu, x, wide) for name, forms in built for gu in (False, True) for x in ("f16", "bf16")
            for wide in (False, True) if not gu or int(forms) & (1 if x == "f16" else 2)}
    want -= {("m4n2w1k8", False, "f16", True), ("m4n2w1k8", True, "f16", True),
             ("m1n4w1k8", False, "bf16", False), ("m1n4w1k8", True, "bf16", False)}
    have = {(tile, gu, x, n >= 4096) for tile, gu, x, _, _, n in _tile_cases()}
    assert want - have == set() and have - want == set()
