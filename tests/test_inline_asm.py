"""CPU: inline assembly of the kernels that loads into a register waits for it in the same statement. To the compiler an assembly
statement's results are there when it ends: of a load that is still in flight it may copy, join or spill the register's old contents,
and nothing tells. Requests whose wait comes later are the compiler's own loads, or go to LDS."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ornith-rs_amd", "csrc")
LOAD = re.compile(r"\b(global_load|buffer_load|flat_load|scratch_load|s_load|s_buffer_load|ds_read|ds_bpermute|ds_permute)\w*")


def _asm_statements(text):
    """the bracketed text of every asm(...) in text"""
    for m in re.finditer(r"\basm\b\s*(?:volatile)?\s*\(", text):
        depth, i, quoted = 1, m.end(), False
        while depth:
            c = text[i]
            if quoted and c == "\\":
                i += 1
            elif c == '"':
                quoted = not quoted
            elif not quoted:
                depth += (c == "(") - (c == ")")
            i += 1
        yield text[m.end():i - 1]


@pytest.mark.parametrize("path", sorted(glob.glob(os.path.join(CSRC, "*.h")) + glob.glob(os.path.join(CSRC, "*.hip"))), ids=os.path.basename)
def test_no_register_is_left_in_flight(path):
    with open(path) as f:
        text = f.read()
    for s in _asm_statements(text):
        m = LOAD.search(s)
        assert not m or "s_waitcnt" in s[m.end():], s
