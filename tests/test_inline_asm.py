"""Inline assembly that writes m0 names it among its clobbers: the compiler may keep a value of its own there."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "loom-skills_amd", "csrc")


def test_asm_that_writes_m0_declares_it():
    blocks = []
    for name in sorted(os.listdir(CSRC)):
        with open(os.path.join(CSRC, name)) as f:
            blocks += [(name, b) for b in re.findall(r"\basm\b[^;]*?\((.*?)\);", f.read(), re.S)]
    writers = [(name, b) for name, b in blocks if re.search(r"s_mov_b32 m0", b)]
    assert writers
    for name, b in writers:
        assert '"m0"' in b, f"{name}: {b}"
