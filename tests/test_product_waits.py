"""The assembly of the tile kernels: nothing but a product reads or writes the
sums of a matrix product too early, on any way through the code.  The hardware
does not wait by itself: a product of 32x32x16 takes 11 other instructions, one
of 32x32x64 19, and the wait at the end of the loop is of 24."""

import re
import shutil
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

from csrc import build as native

WAIT = 24
REG = re.compile(r"\b([av])(?:\[(\d+):(\d+)\]|(\d+)\b)")
LABEL = re.compile(r"([.\w$]+):$")


def _registers(text):
    return {(m[1], i) for m in REG.finditer(text)
            for i in range(int(m[2] or m[4]), int(m[3] or m[4]) + 1)}


def _early(asm):
    """(product, other instruction, instructions between them) within WAIT."""
    code, labels = [], {}
    for line in asm.splitlines():
        line = line.split(";")[0].strip()
        label = LABEL.match(line)
        if label:
            labels[label[1]] = len(code)
        elif re.match(r"[a-z]\w+", line):
            code.append(line)
    products = [i for i, line in enumerate(code) if line.startswith("v_mfma")]
    found = []
    for start in products:
        sums = _registers(code[start].split(",")[0])
        todo, seen = [(start + 1, 0)], set()
        while todo:
            i, passed = todo.pop()
            if i >= len(code) or passed >= WAIT or (i, passed) in seen:
                continue
            seen.add((i, passed))
            op, _, rest = code[i].partition(" ")
            if op == "s_endpgm":
                continue
            if op.startswith(("s_branch", "s_cbranch")):
                todo.append((labels[rest], passed + 1))
            if op == "s_branch":
                continue
            if op.startswith(("v_", "ds_", "global_", "buffer_")) \
                    and _registers(rest) & sums:
                # a product that adds to them waits by itself
                if not op.startswith("v_mfma") or _registers(
                        ",".join(rest.split(",")[1:3])) & sums:
                    found.append((code[start], code[i], passed))
                continue
            todo.append((i + 1, passed + (
                int(rest) + 1 if op == "s_nop" else 1)))
    return len(products), found


def test_the_check_sees_a_missing_wait():
    code = """k:
  v_mfma_f32_32x32x16_bf16 a[0:15], v[0:3], v[4:7], a[0:15]
  s_cbranch_scc1 .L2
  s_branch .L1
.L1:
  s_nop 15
  s_nop 7
  v_accvgpr_read_b32 v8, a15
  s_endpgm
.L2:
  s_nop 3
  v_accvgpr_read_b32 v8, a15
  s_endpgm
"""
    products, early = _early(code)
    assert products == 1 and [(e[1], e[2]) for e in early] == [
        ("v_accvgpr_read_b32 v8, a15", 5)]


@pytest.mark.skipif(not shutil.which(native.HIPCC), reason="no compiler")
def test_sums_of_products_are_waited_for():
    def asm(kernel):
        return subprocess.run(
            [native.HIPCC, "-S", "--cuda-device-only", "-o", "-",
             str(native.CSRC / kernel)] + native.COMMON + native.DEVICE,
            capture_output=True, text=True, check=True).stdout
    kernels = [k.name for k in sorted(native.CSRC.glob("*.hip"))
               if "TileLoop<" in k.read_text()]
    assert len(kernels) >= 2
    with ThreadPoolExecutor(4) as pool:
        for kernel, text in zip(kernels, pool.map(asm, kernels)):
            products, early = _early(text)
            assert products and not early, (kernel, early[:3])


@pytest.mark.skipif(not shutil.which(native.HIPCC), reason="no compiler")
def test_sums_of_wide_tiles_are_waited_for():
    asm = subprocess.run(
        [native.HIPCC, "-S", "--cuda-device-only", "-o", "-",
         str(native.CSRC / "gemm_wide.hip")] + native.COMMON + native.DEVICE,
        capture_output=True, text=True, check=True).stdout
    products, early = _early(asm)
    assert products and not early, early[:3]
