"""What the compiler makes of kernels, where it has been wrong or cannot know: wait states between an instruction and its reader that
hipcc keeps only behind writers that it sees (not in inline assembly), and sums of matrix products in registers that something else gets."""
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


def _lines(text):
    """(operation, operands) of gfx950 assembly; of a label its name and ()"""
    for line in text.splitlines():
        line = line.split(";")[0].strip()
        if line.endswith(":") and " " not in line:
            yield line[:-1], ()
        elif line and not line.startswith("."):
            op, _, rest = line.partition(" ")
            yield op, tuple(x.strip() for x in rest.split(","))


def _is_label(op, operands):
    return not operands


def _early_swaps(text):
    """(writer, swap) pairs less than two wait states apart."""
    found, before = [], []   # before: (wait states, registers written, instruction)
    for op, operands in _lines(text):
        if _is_label(op, operands):
            before = before if op.startswith(".L") else []
            continue
        written = _registers(operands[0]) if op.startswith("v_") else set()
        if op.startswith("v_permlane") and "swap" in op:
            reads, waits = set().union(*map(_registers, operands)), 0
            for states, writes, writer in reversed(before):
                if waits >= 2:
                    break
                if writes & reads:
                    found.append((writer, (op, operands)))
                waits += states
            written = set()   # (a swap behind a swap: the compiler's own)
        before = (before + [(1 + int(operands[0]) if op == "s_nop" else 1, written, (op, operands))])[-4:]
    return found


def _overwritten_sums(text):
    """Matrix products whose sum's registers were not all written by one product before it, or all by something else. Each function is
    gone through in order, and every loop once more with what its end leaves."""
    found, function = [], []

    def follow(at, instruction, writer):
        op, operands = instruction
        if op.startswith("v_mfma"):
            sums = [writer.get(r) for r in _registers(operands[3])]
            products = {w for w in sums if w is not None and w[0].startswith("v_mfma")}
            if products and (len(products) > 1 or any(w not in products for w in sums)):
                found.append(instruction)
        if op.startswith(("v_", "ds_read", "global_load", "buffer_load", "scratch_load")) and not op.startswith(("v_cmp", "v_nop")):
            for r in _registers(operands[0]) | (_registers(operands[1]) if "swap" in op else set()):
                writer[r] = op, at

    def finish():
        writer, labels = {}, {}
        for i, (op, operands) in enumerate(function):
            if _is_label(op, operands):
                labels[op] = i
                continue
            follow(i, (op, operands), writer)
            if op.startswith(("s_branch", "s_cbranch")) and operands[0] in labels:
                again = dict(writer)
                for j in range(labels[operands[0]], i):
                    if not _is_label(*function[j]):
                        follow(j, function[j], again)
        function.clear()

    for op, operands in _lines(text):
        if _is_label(op, operands) and not op.startswith(".L"):
            finish()
        else:
            function.append((op, operands))
    finish()
    return found


def _assembly(source, out):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    subprocess.run([hipcc, "--offload-arch=gfx950", "-O3", "-std=c++17", "-munsafe-fp-atomics", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", f"-I{op_builder.CSRC}/include", "--cuda-device-only", "-S", os.path.join(op_builder.CSRC, source),
                    "-o", str(out)], check=True, capture_output=True)
    return out.read_text()


def test_the_scan_finds_an_early_swap():
    writer, swap, other = "v_cvt_pk_bf16_f32 v15, v15, v30", "v_permlane32_swap_b32_e32 v13, v15", "v_permlane32_swap_b32_e32 v12, v14"
    assert len(_early_swaps(f"{writer}\n{swap}")) == len(_early_swaps(f"{writer}\n{other}\n{swap}")) == 1
    assert len(_early_swaps(f"{writer}\n\ts_nop 0\n{swap}")) == 1
    assert not _early_swaps(f"{writer}\n\ts_nop 1\n{swap}") and not _early_swaps(f"{writer}\n{other}\n\ts_nop 0\n{swap}")


@pytest.mark.parametrize("address,found", [("v[4:5]", True), ("v[6:7]", False)])
def test_the_scan_finds_an_overwritten_sum(address, found):
    text = ["kernel:", "v_mov_b32_e32 v2, 0", "v_mov_b32_e32 v3, 0", "v_mov_b32_e32 v4, 0", "v_mov_b32_e32 v5, 0", ".LBB0_1:",
            f"v_lshl_add_u64 {address}, v[20:21], 0, s[4:5]", f"global_load_dwordx4 v[8:11], {address}, off",
            "v_mfma_f32_16x16x32_bf16 v[2:5], v[8:11], v[12:15], v[2:5]", "s_cbranch_scc1 .LBB0_1", "s_endpgm"]
    assert bool(_overwritten_sums("\n".join(text))) == found


@pytest.mark.skipif(not op_builder.toolchain_available(), reason="needs hipcc")
@pytest.mark.parametrize("source", ["attn/sparse_bwd.hip", "attn/flash_fwd.hip", "attn/flash_small.hip"])
def test_swaps_of_halves_wait_for_their_operands(source, tmp_path):
    """v_permlane*_swap stands two wait states behind a vector write of what it swaps, inline assembly included."""
    text = _assembly(source, tmp_path / "kernels.s")
    assert "v_permlane" in text and not _early_swaps(text)


@pytest.mark.skipif(not op_builder.toolchain_available(), reason="needs hipcc")
@pytest.mark.parametrize("source", ["gemv/skinny_bf16_sh.hip"])
def test_sums_keep_their_registers(source, tmp_path):
    """hipcc 7.2 has put a step's addresses into registers of a product's sums here."""
    text = _assembly(source, tmp_path / "kernels.s")
    assert text.count("v_mfma") > 100 and not _overwritten_sums(text)


def _agprs(operand):
    m = re.fullmatch(r"a(\d+)|a\[(\d+):(\d+)\]", operand.strip())
    if m is None:
        return set()
    return {int(m[1])} if m[1] else set(range(int(m[2]), int(m[3]) + 1))


def _moved_sums(text, after=16, before=2):
    """Accumulators that something other than a product reads fewer than `after` wait states behind the product that wrote them, or that a product
    takes fewer than `before` behind another's write."""
    found, now, product, other = [], 0, {}, {}
    for op, operands in _lines(text):
        if _is_label(op, operands):
            if not op.startswith(".L"):
                product, other = {}, {}
            continue
        now += 1 + int(operands[0]) if op == "s_nop" else 1
        if op.startswith("v_mfma"):
            if any(now - other.get(r, -99) <= before for x in operands[1:] for r in _agprs(x)):
                found.append((op, operands))
            product.update({r: now for r in _agprs(operands[0])})
        elif op.startswith(("v_accvgpr", "scratch_store", "buffer_store", "global_store")):
            read = operands[1:] if op.startswith("v_accvgpr") else operands
            if any(now - product.get(r, -99) <= after for x in read for r in _agprs(x)):
                found.append((op, operands))
            if op.startswith("v_accvgpr"):
                if any(now - product.get(r, -99) <= after for r in _agprs(operands[0])):
                    found.append((op, operands))
                other.update({r: now for r in _agprs(operands[0])})
    return found


def test_the_scan_finds_a_moved_sum():
    product, read, write = "v_mfma_f32_16x16x32_bf16 a[0:3], v[8:11], v[12:15], a[0:3]", "v_accvgpr_read_b32 v2, a3", "v_accvgpr_write_b32 a2, v3"
    assert _moved_sums(f"{product}\n{read}") and _moved_sums(f"{product}\n\ts_nop 7\n{read}") and _moved_sums(f"{write}\n{product}")
    assert _moved_sums(f"{product}\nv_accvgpr_mov_b32 a9, a0") and _moved_sums(f"{product}\n{write}")
    assert not _moved_sums(f"{product}\n\ts_nop 15\n\ts_nop 7\n{read}") and not _moved_sums(f"{write}\n\ts_nop 1\n{product}")


@pytest.mark.skipif(not op_builder.toolchain_available(), reason="needs hipcc")
@pytest.mark.parametrize("source,kernel", [("gemm/wide_gemm.hip", "wide_gemm_kernel"), ("moe/expert_gemm.hip", "expert_big_kernel")])
def test_sums_of_products_in_assembly_stay(source, kernel, tmp_path):
    """The loop of the wide products has them in inline assembly, whose waits hipcc does not know: it must not move, spill or read a sum near one."""
    parts = re.split(r"\n(?=_Z\w+:)", _assembly(source, tmp_path / "kernels.s"))
    text = "\n".join(p.split(".Lfunc_end")[0] for p in parts if kernel in p.split(":")[0])
    assert text.count("v_mfma_f32_16x16x32_bf16 a[") > 1000 and not _moved_sums(text) and not _early_swaps(text)
    assert "scratch_" not in text


@pytest.mark.skipif(not op_builder.toolchain_available(), reason="needs hipcc")
@pytest.mark.parametrize("source", ["attn/flash_dense.hip", "attn/paged_prefill.hip"])
def test_swaps_of_results_wait_for_their_operands(source, tmp_path):
    text = _assembly(source, tmp_path / "kernels.s")
    assert "v_permlane16_swap" in text and not _early_swaps(text)
