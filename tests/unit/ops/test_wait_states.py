"""Wait states that hipcc keeps between an instruction and its reader, and cannot keep where the writer is inline assembly."""
import os
import re
import shutil
import subprocess

import pytest

from deepspeedsyclsupport_amd.ops import op_builder


def _registers(operand):
    m = re.fullmatch(r"v(\d+)|v\[(\d+):(\d+)\]", operand.strip())
    if m is None:
        return set()
    return {int(m[1])} if m[1] else set(range(int(m[2]), int(m[3]) + 1))


def _early_swaps(text):
    """(writer, swap) pairs less than two wait states apart in gfx950 assembly."""
    found, before = [], []   # before: (wait states, registers written, line)
    for line in text.splitlines():
        line = line.split(";")[0].strip()
        if not line or line.startswith("."):
            continue
        if line.endswith(":"):
            before = [] if not line.startswith(".L") else before
            continue
        op, _, rest = line.partition(" ")
        operands = rest.split(",")
        if op.startswith("v_permlane") and "swap" in op:
            reads, waits = set().union(*map(_registers, operands)), 0
            for states, written, writer in reversed(before):
                if waits >= 2:
                    break
                if written & reads:
                    found.append((writer, line))
                waits += states
            written = set()   # (a swap behind a swap: the compiler's own)
        else:
            written = _registers(operands[0]) if op.startswith("v_") else set()
        before = (before + [(1 + int(operands[0]) if op == "s_nop" else 1, written, line)])[-4:]
    return found


def test_the_scan_finds_an_early_swap():
    writer, swap = "v_cvt_pk_bf16_f32 v15, v15, v30", "v_permlane32_swap_b32_e32 v13, v15"
    other = "v_permlane32_swap_b32_e32 v12, v14"
    assert _early_swaps(f"{writer}\n{swap}") == _early_swaps(f"{writer}\n{other}\n{swap}") == [(writer, swap)]
    assert _early_swaps(f"{writer}\n\ts_nop 0\n{swap}") == [(writer, swap)]
    assert not _early_swaps(f"{writer}\n\ts_nop 1\n{swap}") and not _early_swaps(f"{writer}\n{other}\n\ts_nop 0\n{swap}")


@pytest.mark.skipif(not op_builder.toolchain_available(), reason="needs hipcc")
@pytest.mark.parametrize("source", ["attn/sparse_bwd.hip", "attn/flash_fwd.hip", "attn/flash_small.hip"])
def test_swaps_of_halves_wait_for_their_operands(source, tmp_path):
    """v_permlane*_swap stands two wait states behind a vector write of what it swaps, inline assembly included."""
    out = tmp_path / "kernels.s"
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    subprocess.run([hipcc, "--offload-arch=gfx950", "-O3", "-std=c++17", "-munsafe-fp-atomics", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", f"-I{op_builder.CSRC}/include", "--cuda-device-only", "-S", os.path.join(op_builder.CSRC, source),
                    "-o", str(out)], check=True, capture_output=True)
    text = out.read_text()
    assert "v_permlane" in text and not _early_swaps(text)
