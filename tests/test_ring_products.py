"""Products written in assembly (ring_gemm.h) get no wait states from the compiler: in the built
kernels nothing but the products touches a sum between the first and the last of them, and a
fragment comes from LDS, not from another vector instruction right ahead of its product."""

from __future__ import annotations

import os
import re
import shutil
import subprocess
from pathlib import Path

import pytest

ROCM = Path(os.environ.get("ROCM_PATH", "/opt/rocm"))
PACKAGE = Path(__file__).resolve().parent.parent / "vllm_tgis_adapter_amd"
OBJDUMP = shutil.which("llvm-objdump", path=f"{ROCM}/llvm/bin:{os.environ.get('PATH', '')}")
PRODUCT = "v_mfma_f32_16x16x32_bf16"


def _registers(operand: str) -> set[int]:
    found = re.fullmatch(r"v\[(\d+):(\d+)\]|v(\d+)", operand.strip())
    if not found:
        return set()
    if found[3]:
        return {int(found[3])}
    return set(range(int(found[1]), int(found[2]) + 1))


def _kernels(name: str, tmp_path: Path):
    shutil.copy(PACKAGE / name, tmp_path / name)
    subprocess.run([OBJDUMP, "--offloading", name], cwd=tmp_path, check=True, capture_output=True)
    for code in sorted(tmp_path.glob(f"{name}.*gfx950")):
        listing = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", code],
                                 check=True, capture_output=True, text=True).stdout
        for part in re.split(r"^<(?=\w*(?:_ring_kernel|gemm_ring_lora))", listing, flags=re.M)[1:]:
            lines = [line.split("//")[0].strip() for line in part.splitlines()]
            end = lines.index("") if "" in lines else len(lines)
            kernel, body = lines[0].rstrip(">:"), lines[1:end]
            if tile := re.search(r"gemm_ring_loraILi(\d+)ELi(\d+)E", kernel):
                body = _beside_a_shrink(kernel, body, int(tile[1]) * int(tile[2]) // 256)
            yield kernel, body


def _beside_a_shrink(kernel: str, body: list[str], products: int) -> list[str]:
    """The part of a kernel that makes a tile's products: a round of the loop has two of 16 x 16 and
    64 inputs, each two products, by four waves.  The other part, the adapters' shrink, has eight
    of the compiler's own."""
    parts = [[]]
    for line in body:
        parts[-1].append(line)
        if line.startswith("s_endpgm"):
            parts.append([])
    counts = [sum(line.startswith(PRODUCT) for line in part) for part in parts]
    assert sorted(n for n in counts if n) == [8, products], (kernel, counts)
    return parts[counts.index(products)]


@pytest.mark.skipif(OBJDUMP is None, reason="no llvm-objdump")
@pytest.mark.parametrize(("name", "least"), [("_C.so", 38), ("_C_seq.so", 12)])
def test_sums_and_fragments_stay_in_place(name, least, tmp_path):
    if not (PACKAGE / name).exists():
        pytest.skip("the extension is not built")
    kernels = 0
    for kernel, body in _kernels(name, tmp_path):
        at = [i for i, line in enumerate(body) if line.startswith(PRODUCT)]
        assert at, kernel
        kernels += 1
        for line in body[at[0]:at[-1]]:
            assert "accvgpr" not in line and "scratch_" not in line, (kernel, line)
        for i in at:
            to, a, b, c = (o.strip() for o in body[i][len(PRODUCT):].split(",")[:4])
            assert to == c and c.startswith("a["), (kernel, body[i])
            # two wait states lie between a vector instruction and the product that reads what
            # it wrote; here four instructions, whatever they are
            read = _registers(a) | _registers(b)
            assert len(read) in (4, 8), (kernel, body[i])
            for line in body[max(0, i - 4):i]:
                if line.startswith("v_") and not line.startswith((PRODUCT, "v_cmp")):
                    wrote = _registers(line.split(None, 1)[1].split(",")[0])
                    assert not read & wrote, (kernel, line, body[i])
        # what reads a sum first waits for the last product
        behind = body[at[-1] + 1:]
        behind = behind[:next(i for i, line in enumerate(behind) if re.search(r"\ba\[?\d", line))]
        waits = sum(int(line.split()[1], 0) + 1 if line.startswith("s_nop") else 1
                    for line in behind)
        assert waits >= 18, (kernel, behind)
    assert kernels >= least


@pytest.mark.skipif(OBJDUMP is None, reason="no llvm-objdump")
def test_a_large_panel_computes_no_places_for_its_loads(tmp_path):
    """In int8 panels of 160 x 256 (gemm_panel_q.h) a wave is alone on its SIMD, and every instruction
    beyond those that hide behind the products takes its four clocks: a load's place in LDS is a
    register and a literal, one instruction each.  (Of remainders, copied: 282 instructions.)"""
    if not (PACKAGE / "_C.so").exists():
        pytest.skip("the extension is not built")
    shutil.copy(PACKAGE / "_C.so", tmp_path / "_C.so")
    subprocess.run([OBJDUMP, "--offloading", "_C.so"], cwd=tmp_path, check=True,
                   capture_output=True)
    loops = []
    for code in sorted(tmp_path.glob("_C.so.*gfx950")):
        listing = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", code],
                                 check=True, capture_output=True, text=True).stdout
        for part in re.split(r"^\w+ <(?=\w*gemm_panel_q_kernelILi8ELi10ELi4E)", listing,
                             flags=re.M)[1:]:
            found = re.findall(r"^\s+(\w[^/]*?)\s*// ([0-9A-F]+):", part.split("\n\n")[0], flags=re.M)
            at = {int(address, 16): i for i, (_, address) in enumerate(found)}
            for i, (line, address) in enumerate(found):
                if branch := re.match(r"s_cbranch\w* (\d+)", line):
                    words = (int(branch[1]) ^ 0x8000) - 0x8000   # of 16 bits, from behind it on
                    loop = [line for line, _ in found[at.get(int(address, 16) + 4 + 4 * words, i):i + 1]]
                    if sum(line.startswith(PRODUCT) for line in loop) == 80:
                        loops.append(loop)
    assert len(loops) == 2   # without and with the gate
    for loop in loops:
        assert sum(line.startswith("buffer_load") for line in loop) == 9
        assert len(loop) <= 272, "\n".join(loop)
