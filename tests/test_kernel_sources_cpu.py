"""Rules that the kernel sources keep, checked on their text."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dynaflow_amd", "csrc")
ASM = re.compile(r"\basm\b\s*(?:volatile)?\s*\(((?:[^()\"]|\"(?:[^\"\\]|\\.)*\"|\([^()]*\))*)\)", re.S)
LOAD = re.compile(r"\b(?:global|flat|buffer|scratch|s|s_buffer)_load_(?!lds)\w+|\bds_read\w*")


def asm_loads_into_registers(text):
    return [m.group(0) for m in ASM.finditer(text)
            if LOAD.search(m.group(1)) and "=" in m.group(1) and "waitcnt" not in m.group(1)]


def test_no_load_in_inline_assembly_leaves_its_wait_to_another_statement():
    """The compiler takes the output registers of an asm statement as written when the statement has been issued: it may
    copy them, or give them to something else where the value is not used, while the load is still on its way."""
    split = 'asm volatile("global_load_dwordx4 %0, %1, off sc1" : "=v"(v) : "v"(p) : "memory");'
    assert asm_loads_into_registers(split)
    assert not asm_loads_into_registers(split.replace(" sc1", " sc1\\n\\ts_waitcnt vmcnt(0)"))
    assert not asm_loads_into_registers('asm volatile("s_mov_b32 m0, %0\\n\\tglobal_load_lds_dwordx4 %1, off" ::"s"(a), "v"(g));')
    sources = glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.h"))
    assert len(sources) >= 9
    for path in sources:
        with open(path) as f:
            assert not asm_loads_into_registers(f.read()), path
