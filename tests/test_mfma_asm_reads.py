"""Static check of the asm statements that read results of matrix products in the prompt attention kernel's machine code.

The hardware does not wait when an instruction reads the registers of a matrix product that has not finished, and the compiler puts
the cycles it needs in front of its own instructions only, not in front of a source's asm statements.  So between a product and the
first asm instruction that reads one of its registers there has to be an instruction of the compiler's that reads one: it stands
behind the wait.  (Instructions in the order they are written; a kernel's text is followed twice, for loops.)
"""
import re
import shutil
from pathlib import Path

import pytest

from test_wait_counts import CSRC, _assembly, _kernels

REGS = re.compile(r"\bv(?:\[(\d+):(\d+)\]|(\d+)\b)")


def _registers(operand: str):
    m = REGS.search(operand)
    return set() if not m else {int(m.group(3))} if m.group(3) else set(range(int(m.group(1)), int(m.group(2)) + 1))


def _unguarded_reads(lines):
    """(instructions that read a product's registers from inside an asm statement, those of them that nothing of the compiler's
    read the same product before)"""
    pending, reads, bad = [], [], []  # pending: registers of products that no instruction of the compiler's has read yet
    for line, inline in lines + lines:
        op, _, rest = line.partition(" ")
        if not op.startswith(("v_", "ds_", "buffer_", "global_", "flat_")) or op.startswith("v_nop"):
            continue
        operands = rest.split(",")
        # (a store's operands are all sources)
        dst = set() if "store" in op or op.startswith("ds_write") else _registers(operands[0])
        src = set().union(*[_registers(o) for o in (operands if not dst else operands[1:])], set())
        if op.startswith("v_mfma"):
            # (a product that takes another's result as its third operand is waited for by the compiler)
            pending = [p for p in pending if not p & src] + [dst]
            continue
        hit = [p for p in pending if p & src]
        if inline:
            reads.append(line)
            bad += [line] if hit else []
        else:
            pending = [p for p in pending if not p & src]
    return reads, bad


def test_asm_statements_read_no_product_that_nothing_has_waited_for(tmp_path):
    if shutil.which("hipcc") is None and not Path("/opt/rocm/bin/hipcc").exists():
        pytest.skip("hipcc not available")
    kernels = list(_kernels(_assembly(CSRC / "gptq4_attention.hip", tmp_path)))
    assert len(kernels) == 1
    reads, bad = _unguarded_reads(kernels[0][1])
    assert sum(l.startswith("v_max3_f32") for l in reads) >= 30  # (the scan sees them)
    assert not bad, bad


def test_the_scan_sees_a_read_without_a_wait():
    product = ("v_mfma_f32_32x32x16_f16 v[0:15], v[20:23], v[24:27], v[0:15]", False)
    asm = ("v_max3_f32 v30, v30, v3, v31", True)
    assert _unguarded_reads([product, asm])[1]
    assert _unguarded_reads([product, ("v_max_f32_e32 v32, v5, v5", False), asm, ("v_mov_b32_e32 v0, 0", False)])[1] == []
    assert _unguarded_reads([product, ("v_max_f32_e32 v5, v32, v32", False), asm])[1]  # (a write is no read)
