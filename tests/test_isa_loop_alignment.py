"""Where the tile loop of the decode kernel lies does not depend on what stands in front of it: most of its 8-byte instructions begin
at a multiple of 8 bytes, also with one 4-byte instruction more at the kernel's first line."""
import os
import re
import shutil
import subprocess

import pytest

from yasakani_amd import isa_check

LLVM = os.path.join(os.path.dirname(os.path.dirname(isa_check.HIPCC)), "llvm", "bin")


def loop_instructions(listing):
    """(address, bytes) of what lies between the two waits of the tile loop (the last two waits that leave one tile in flight), per kernel"""
    kernels, cur = {}, None
    for line in listing.split("\n"):
        m = re.match(r"^[0-9a-f]+ <(_Z\w+)>:", line)
        if m:
            cur = kernels.setdefault(m.group(1), [])
            continue
        m = re.search(r"// ([0-9A-F]{12}): ([0-9A-F ]+)", line)
        if m and cur is not None:
            cur.append((int(m.group(1), 16), 4 * len(m.group(2).split()), "vmcnt(16)" in line))
    out = {}
    for name, ins in kernels.items():
        waits = [n for n, x in enumerate(ins) if x[2]]
        if "attend_narrow_kernel" in name and len(waits) >= 2:
            out[name] = [x[:2] for x in ins[waits[-2]:waits[-1]]]
    return out


@pytest.mark.skipif(shutil.which(isa_check.HIPCC) is None and not os.path.exists(isa_check.HIPCC), reason="hipcc not found")
def test_decode_loop_keeps_its_alignment(tmp_path):
    asm, moved, obj = (str(tmp_path / n) for n in ("a.s", "b.s", "b.o"))
    subprocess.run([isa_check.HIPCC, *isa_check.FLAGS, *isa_check.EXTRA["attend_narrow.hip"], "attend_narrow.hip", "-o", asm], cwd=isa_check.CSRC, check=True)
    with open(asm) as f:
        text = f.read()
    # the first line behind the entry that fetches the preloaded arguments where the hardware has not
    entry = re.compile(r"(\.p2align\t8\n(?:;[^\n]*\n)*\.LBB\d+_\d+:[^\n]*\n)")
    assert len(entry.findall(text)) >= 2
    for extra in (0, 1):
        with open(moved, "w") as f:
            f.write(entry.sub(lambda m: m.group(1) + "\ts_nop 0\n" * extra, text))
        subprocess.run([os.path.join(LLVM, "clang"), "-target", "amdgcn-amd-amdhsa", "-mcpu=gfx950", "-c", moved, "-o", obj], check=True)
        listing = subprocess.run([os.path.join(LLVM, "llvm-objdump"), "-d", obj], check=True, capture_output=True, text=True).stdout
        loops = loop_instructions(listing)
        assert len(loops) == 2, sorted(loops)              # single-stream and multi-stream
        for name, ins in loops.items():
            wide = [a for a, n in ins if n == 8]
            assert len(wide) > 100
            assert sum(a % 8 == 0 for a in wide) > 0.6 * len(wide), (name, extra)
