"""The combiners that ask for everything in one trip to memory do: in the generated code no wait for a load stands in front of the last request
of a step (left alone the compiler sinks requests behind uses of earlier answers)."""
import os
import re
import shutil
import subprocess

import pytest

from yasakani_amd import isa_check

# kernel name, 16-byte requests of a step, 4-byte requests of a step: one entry per step
FORMS = [("attend_narrow.hip", "combine_rows_kernelILb0E", [(8, 2)]),
         ("attend_narrow.hip", "combine_rows_kernelILb1E", [(1, 2), (2, 2), (4, 2), (8, 2), (8, 16)]),
         ("attend_narrow.hip", "combine_kernelILi1ELb0ELb0E", [(4, 2)]),
         ("attend_narrow.hip", "combine_kernelILi4ELb0ELb0E", [(16, 8)]),
         ("attend256.hip", "combine256_kernelILi4ELi1ELb0ELi0E", [(4, 2)]),
         ("attend256.hip", "combine256_kernelILi8ELi2ELb0ELi0E", [(16, 8)])]


def steps(lines):
    """Per straight run of code with 16-byte loads: (16-byte loads, 4-byte loads, loads that a wait for a load stands in front of)."""
    out, block, waited = [], [0, 0, 0], False
    for raw in lines + [".L:"]:
        t = raw.split(";")[0].strip()
        if re.match(r"\.L\w*:", t) or t.startswith(("s_cbranch", "s_branch", "s_endpgm")):
            if block[0]:
                out.append(tuple(block))
            block, waited = [0, 0, 0], False
        elif t.startswith("global_load_dword"):
            block[0 if t.startswith("global_load_dwordx4") else 1] += 1
            block[2] += waited
        elif t.startswith("s_waitcnt") and "vmcnt" in t:
            waited = True
    return out


def test_steps_counts_what_comes_late():
    listing = """
	global_load_dword v1, v2, s[4:5]
	global_load_dwordx4 v[4:7], v2, s[4:5]
	s_waitcnt vmcnt(1)
	global_load_dword v3, v2, s[6:7]
	s_waitcnt vmcnt(0)
.LBB0_1:
	global_load_dwordx4 v[4:7], v2, s[4:5]
	s_endpgm
"""
    assert steps(listing.split("\n")) == [(1, 2, 1), (1, 0, 0)]


@pytest.mark.skipif(shutil.which(isa_check.HIPCC) is None and not os.path.exists(isa_check.HIPCC), reason="hipcc not found")
def test_no_wait_in_front_of_the_last_request(tmp_path):
    kernels = {}
    for src in sorted({f[0] for f in FORMS}):
        out = str(tmp_path / (src + ".s"))
        subprocess.run([isa_check.HIPCC, *isa_check.FLAGS, *isa_check.EXTRA[src], src, "-o", out], cwd=isa_check.CSRC, check=True)
        with open(out) as f:
            kernels.update({(src, name): lines for name, lines in isa_check.kernels_of(f.read())})
    for src, part, want in FORMS:
        found = [lines for (s, name), lines in kernels.items() if s == src and part in name]
        assert len(found) == 1, part
        assert sorted(steps(found[0])) == sorted((a, b, 0) for a, b in want), part
