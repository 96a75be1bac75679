"""Where the lanes of a divergent branch meet again, the block begins by
switching the others back on (s_or_b64 exec, exec, ...).  hipcc 7.2 has put
constants and copies back into vector registers before that instruction, in the
FP64 table-driven kernel for 16 x 16 with its 434 registers: lanes that had
skipped the branch went on with what the register held, and a simulation never
ended.  The library's kernels are compiled to assembly here and searched for
that (no GPU needed)."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "py_stoch_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
VECTOR_WRITE = re.compile(r"v_(?!cmp|readlane|readfirst|writelane|nop)|(global|ds|scratch|flat|buffer)_(load|read)")
END = re.compile(r"s_\w+_b64 exec,|s_\w*saveexec|s_cbranch|s_branch|s_swappc|s_setpc|s_endpgm")


def early_writes(text):
    """Vector writes at the head of a block that lanes skip to, before it
    restores exec: [(label, [instructions])]."""
    lines = text.split("\n")
    targets = set(re.findall(r"s_cbranch_execz (\.LBB\w+)", text))
    out = []
    for i, line in enumerate(lines):
        m = re.match(r"(\.LBB\w+):", line)
        if not m or m.group(1) not in targets:
            continue
        writes = []
        for l in lines[i + 1:]:
            if re.match(r"\.LBB|; %bb", l):
                break
            ins = l.split(";")[0].strip()
            if not ins:
                continue
            if END.match(ins):
                if writes and re.match(r"s_or_b64 exec, exec, s", ins):
                    out.append((m.group(1), writes))
                break
            if VECTOR_WRITE.match(ins):
                writes.append(ins)
    return out


def test_the_search_finds_a_planted_write():
    good = "\ts_cbranch_execz .LBB0_2\n; %bb.1:\n\tv_mov_b32_e32 v1, 0\n.LBB0_2:\n\ts_or_b64 exec, exec, s[0:1]\n\tv_mov_b32_e32 v2, 1.0\n"
    assert early_writes(good) == []
    bad = good.replace(".LBB0_2:\n", ".LBB0_2:\n\tv_mov_b32_e32 v3, 0x3ff00000\n")
    assert early_writes(bad) == [(".LBB0_2", ["v_mov_b32_e32 v3, 0x3ff00000"])]


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is not installed")
@pytest.mark.parametrize("source,extra", [("pst_fp64.hip", ["-ffp-contract=off"]), ("pst_mixed.hip", []),
                                          ("pst_wave.hip", [])])
def test_no_vector_write_before_the_lanes_are_back(tmp_path, source, extra):
    out = tmp_path / "kernels.s"
    subprocess.run([HIPCC, *FLAGS, *extra, "--offload-device-only", "-S", os.path.join(CSRC, source), "-o", str(out)],
                   check=True, stderr=subprocess.DEVNULL)
    assert early_writes(out.read_text()) == []
