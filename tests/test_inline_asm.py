"""What the inline assembly of the kernels tells the compiler."""
import glob
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def asm_statements():
    for path in sorted(glob.glob(os.path.join(ROOT, "pimaicompiler_amd", "csrc", "*.h*"))):
        for m in re.finditer(r"asm volatile\((.*?)\);", open(path).read(), flags=re.S):
            yield os.path.basename(path), m.group(1)


def test_a_statement_that_writes_m0_says_so():
    writes = [(f, a) for f, a in asm_statements() if re.search(r"s_mov_b32 m0", a)]
    assert writes
    assert all(re.search(r':[^:]*"m0"[^:]*$', a) for _, a in writes), writes
