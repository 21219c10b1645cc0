"""Inline assembly in the device code, on the CPU.

m0 and exec are reserved: the compiler need not honour them in a clobber list
(it says so on each build), so an asm block has to leave them as it found them.
Every instruction that writes m0 stands between one that saves it to a register
operand and one that puts it back.
"""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mosaic-art-rust_amd", "csrc")


def test_reserved_registers_are_not_clobbered():
    for path in sorted(glob.glob(os.path.join(CSRC, "*.h*"))):
        text = open(path).read()
        assert not re.search(r'"(m0|exec)"\s*[,)]', text), path
        writes = re.findall(r"s_[a-z]+_[bu]32 m0, ([^\\]+)\\n", text)
        if not writes:
            continue
        save = re.search(r"s_mov_b32 (%\[\w+\]), m0\\ns_mov_b32 m0, ", text)
        assert save, path
        assert f"s_mov_b32 m0, {save.group(1)}\\n" in text, path
