"""The built kernels' instructions: what the matrix cores' results ask of the instructions behind them (no GPU).

The cores' results are not interlocked. The compiler keeps their distances where it knows both instructions, and not all of them.
"""

from __future__ import annotations

import re
import shutil
import subprocess
from typing import NamedTuple, Optional

import pytest

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


class Instruction(NamedTuple):
    kernel: str
    address: int
    op: str
    operands: list[str]


def _registers(operand: str) -> Optional[tuple[int, int]]:
    m = re.match(r"-?\|?v\[?(\d+)(?::(\d+))?\]?", operand)
    return (int(m.group(1)), int(m.group(2) or m.group(1))) if m else None


def _overlap(a: Optional[tuple[int, int]], b: Optional[tuple[int, int]]) -> bool:
    return a is not None and b is not None and a[0] <= b[1] and b[0] <= a[1]


@pytest.fixture(scope="module")
def listing(tmp_path_factory):
    """The instructions of the kernels that use the matrix cores, in their order."""
    if shutil.which(OBJDUMP) is None:
        pytest.skip("needs the ROCm toolchain's disassembler")
    from dli_amd.kernels import build

    folder = tmp_path_factory.mktemp("listing")
    shutil.copy(build.find_library() or build.build(), folder / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=folder, check=True, capture_output=True)
    instructions = []
    for code in sorted(folder.glob("lib.so.*amdgcn*")):
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", code.name], cwd=folder, check=True, capture_output=True, text=True).stdout
        for block in text.split("\n\n"):
            if "v_mfma" not in block:
                continue
            kernel = re.search(r"<(.*)>:", block).group(1) + code.name
            for line in block.splitlines():
                instruction, _, place = line.partition("//")
                op, _, rest = instruction.strip().partition(" ")
                if place:
                    operands = [o.split(" ")[0] for o in rest.strip().split(", ")]
                    instructions.append(Instruction(kernel, int(place.split(":")[0], 16), op, operands))
    assert sum(i.op.startswith("v_mfma") for i in instructions) > 1000
    return instructions


def test_no_product_adds_to_one_of_another_depth(listing):
    """A product that takes the sum of a product of another depth right behind it has read that sum before it was there, and the
    compiler inserts no wait: nothing may depend on what happens to stand between the two."""
    found, sums, kernel = set(), {}, ""
    for i in listing:
        if i.kernel != kernel:
            sums, kernel = {}, i.kernel
        if not i.op.startswith("v_mfma"):
            written = _registers(i.operands[0]) if i.op.startswith(("v_", "ds_read", "buffer_load", "global_load")) else None
            if written is not None:
                sums = {r: op for r, op in sums.items() if not _overlap(r, written)}
            continue
        taken, written = _registers(i.operands[3]), _registers(i.operands[0])
        if taken is not None and sums.get(taken, i.op) != i.op:
            found.add((i.kernel, i.op, sums[taken]))
        sums = {r: op for r, op in sums.items() if not _overlap(r, written)}
        if written is not None:
            sums[written] = i.op
    assert not found


def test_vector_instructions_wait_for_a_products_result(listing):
    """A vector instruction that reads the result of a 16x16x16 or 16x16x32 product stands at least seven wait states (an
    instruction each, s_nop n another n) behind it on every way there, branches taken included."""
    apart = 7
    at = {(i.kernel, i.address): n for n, i in enumerate(listing)}
    found = set()
    for n, product in enumerate(listing):
        if not product.op.startswith(("v_mfma_f32_16x16x16_bf16", "v_mfma_f32_16x16x32_bf16")):
            continue
        result, ways, seen = _registers(product.operands[0]), [(n + 1, 0)], {}
        while ways:
            j, states = ways.pop()
            if j >= len(listing) or states >= apart or seen.get(j, apart) <= states:
                continue
            seen[j] = states
            i = listing[j]
            if i.op.startswith("v_mfma"):
                if _overlap(_registers(i.operands[0]), result):
                    continue   # (another product's result from here on)
            elif i.op.startswith("v_") and any(_overlap(_registers(o), result) for o in i.operands[1:]):
                found.add((i.kernel, i.op, states))
                continue
            if i.op in ("s_endpgm", "s_setpc_b64"):
                continue
            if i.op.startswith("s_cbranch") or i.op == "s_branch":
                words = int(i.operands[0])
                ways.append((at[i.kernel, i.address + 4 + 4 * (words - 65536 if words > 32767 else words)], states + 1))
                if i.op == "s_branch":
                    continue
            ways.append((j + 1, states + 1 + (int(i.operands[0]) if i.op == "s_nop" else 0)))
    assert not found


def test_a_merge_of_runs_asks_for_all_of_them_at_once(listing):
    """The decode attention's workgroup that merges eight or sixteen runs has what all of them left on its way before it waits for
    the first: a load of four sums and one of two statistics each (of which the compiler takes a pair or two as one)."""
    most, asked = {}, 0
    for i in listing:
        kernel = re.search(r"attention_decode_kernelILi(\d+)ELi(\d+)ELi(\d+)E", i.kernel)
        if kernel is None:
            continue
        kernel = tuple(map(int, kernel.groups()))
        if i.op.startswith("buffer_load"):
            asked += 1
        elif i.op == "s_waitcnt" and any(o.startswith("vmcnt") for o in i.operands):
            most[kernel], asked = max(most.get(kernel, 0), asked), 0
    # (sixteenths of a head, waves, runs): heads of up to 48 have a copy for eight runs
    assert set(most) == {(d, w, r) for d in range(1, 9) for w in (4, 8) for r in ((8, 16) if d <= 3 else (16,))}
    assert all(n >= 2 * r - 2 for (_, _, r), n in most.items()), most
