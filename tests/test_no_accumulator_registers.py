"""Kernels whose score products start in inline asm keep them in ordinary registers.

The compiler does not know that the asm holds a matrix instruction.  Were its results to be moved to accumulation registers right behind
it, as happens when a kernel may use more than 256 registers, nothing would keep the moves from reading them too early."""
import re
import subprocess

from test_lds_read_windows import OBJDUMP, code_objects, functions, kernels, LIB  # noqa: F401


def test_no_accumulation_registers(kernels):                     # noqa: F811
    seen = 0
    for obj in code_objects(LIB):
        if b"block_sparse_attn_kernel" not in obj:
            continue
        asm = subprocess.run([OBJDUMP, "-d", "-"], input=obj, capture_output=True).stdout.decode()
        for name, code in functions(asm).items():
            if not any(op == "v_mfma_i32_32x32x32_i8" for _, op, _, _ in code):
                continue
            seen += 1
            assert not any("accvgpr" in op or re.search(r"\ba(\d|\[)", ops) for _, op, ops, _ in code), name
    assert seen >= 80
