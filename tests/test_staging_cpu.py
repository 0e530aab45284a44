"""CPU test of how the kernels' sources form buffer loads: every row beyond a descriptor's end
reads zeros because its *per-lane* offset (the instruction's immediate with it) is past the
descriptor's bytes.  The instruction's scalar offset is not part of that comparison in a way
this code may rest on, so no buffer load uses one: a query row past the last one, or a key past
a sequence's end, moved there would be read from the memory behind the tensor.
"""

from __future__ import annotations

import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mla-cuda_amd",
                    "csrc")


def sources():
    for path in sorted(glob.glob(os.path.join(CSRC, "*.h")) + glob.glob(os.path.join(CSRC, "*.hip"))):
        with open(path) as f:
            yield os.path.basename(path), re.sub(r"//[^\n]*", "", f.read())


def test_buffer_loads_have_no_scalar_offset():
    asm, builtin = [], []
    for name, text in sources():
        # buffer_load_dwordx4 vaddr, srsrc, soffset offen ...: 0, or an operand bound to 0u
        for m in re.finditer(r"buffer_load_\w+ %\d, %\d, (\S+) offen[^;]*;", text):
            soff = m.group(1)
            if soff.startswith("%"):
                inputs = re.findall(r'"\w"\(([^()]*)\)', m.group(0))
                soff = inputs[int(soff[1:])]
            asm.append((name, m.group(0), soff))
        builtin += [(name, m.group(0), m.group(1).strip())
                    for m in re.finditer(r"raw_buffer_load_\w+\(\w+, [^;]*?, ([^,;]+), \w+\)", text)]
    assert len(asm) >= 2 and builtin
    assert [x for x in asm + builtin if x[2] not in ("0", "0u")] == []
