"""Rules of the gfx950 instruction set that the compiler keeps for its own instructions and cannot keep for
inline assembly, checked on the assembly of the device sources (compiled here, without a GPU)."""
import re
import subprocess
import sys
from pathlib import Path

import pytest

REPO = Path(__file__).resolve().parents[1]
PKG = REPO / "unified-memory-scheduler_amd"


@pytest.fixture(scope="module")
def device_asm(tmp_path_factory):
    """name -> the instructions of a device source, in order, with the marks around inline assembly."""
    sys.path.insert(0, str(PKG))
    import build_lib
    cache = {}

    def lines(name):
        if name not in cache:
            out = tmp_path_factory.mktemp("asm") / (name + ".s")
            cmd = [build_lib.hipcc(), *build_lib.HIP_FLAGS, f"-I{build_lib.HOST}", "-x", "hip", "-S", "--cuda-device-only",
                   str(build_lib.CSRC / name), "-o", str(out)]
            proc = subprocess.run(cmd, capture_output=True, text=True)
            assert proc.returncode == 0, proc.stderr
            text = [line.strip() for line in out.read_text().splitlines()]
            cache[name] = [line for line in text if line.startswith(";;#ASM") or re.match(r"[svgd][a-z0-9]*_|buffer_|flat_|scratch_", line)]
        return cache[name]

    return lines


def wait_states(instruction):
    m = re.match(r"s_nop (\d+)", instruction)
    return int(m.group(1)) + 1 if m else 1


def test_loads_to_lds_are_a_wait_state_behind_their_m0_write(device_asm):
    """A load to LDS takes its address from M0 and needs one wait state behind a scalar write of it."""
    since, loads, bad = 99, 0, []
    for line in device_asm("vbm_gemm.hip"):
        if line.startswith(";;"):
            continue
        if "_load_lds_" in line or re.match(r"buffer_load.*\blds\b", line):
            loads += 1
            if since < 1:
                bad.append(line)
        since = 0 if re.match(r"s_\w+ m0,", line) else since + wait_states(line)
    assert loads > 0
    assert not bad, (len(bad), bad[:3])


def registers(operand):
    m = re.match(r"v\[(\d+):(\d+)\]|v(\d+)\b", operand.strip())
    if not m:
        return set()
    return set(range(int(m.group(1)), int(m.group(2)) + 1)) if m.group(1) else {int(m.group(3))}


def test_matrix_results_stay_whole_until_the_inline_sum_that_reads_them(device_asm):
    """A matrix instruction writes its registers some wait states late. The compiler keeps its own writes to
    a result's free lanes apart from that, and inline assembly's not: a result that an inline sum reads has to
    keep all its lanes up to the sum."""
    pending, sums, bad, inline = [], 0, [], False
    for line in device_asm("vbm_gemv.hip"):
        if line.startswith(";;"):
            inline = line.startswith(";;#ASMSTART")
            continue
        op, _, rest = line.partition(" ") if " " in line else line.partition("\t")
        operands = re.split(r",(?![^\[]*\])", rest)
        writes = registers(operands[0]) if re.match(r"v_(?!cmp)|ds_read|buffer_load|global_load|scratch_load", op) else set()
        reads = set().union(*(registers(o) for o in operands[1:]))
        for result in pending[:]:
            if reads & result["regs"]:
                if inline:
                    sums += 1
                    bad += [result["line"]] if result["lost"] else []
                pending.remove(result)
            elif writes & result["regs"]:
                result["lost"] = True
        if op.startswith("v_mfma_f32_4x4x4"):
            pending.append({"line": line, "regs": writes, "lost": False})
            del pending[:-8]
    assert sums > 0
    assert not bad, (len(bad), bad[:3])
