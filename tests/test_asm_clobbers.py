"""Inline asm of the kernels: a statement that writes a fixed scalar register (m0, vcc, exec, scc by s_cmp) names it as
clobbered, since the compiler keeps values of its own there. CPU only: reads the sources."""
import glob
import os
import re

from conftest import PKG

FIXED = {r"\b(?:s_mov_b32|s_add_u32|s_movk_i32)\s+m0\b": "m0", r"\bs_mov_b64\s+vcc\b": "vcc", r"\bv_cmp\w*\s+vcc\b": "vcc",
         r"\bs_mov_b64\s+exec\b": "exec", r"\bs_cmp_": "scc"}


def asm_statements(text):
    """The argument lists of the asm statements (from "asm volatile(" to its closing parenthesis)."""
    for m in re.finditer(r"\basm\s*(?:volatile\s*)?\(", text):
        depth, i, quoted = 1, m.end(), False
        while depth:
            c = text[i]
            if c == "\\" and quoted:
                i += 1
            elif c == '"':
                quoted = not quoted
            elif not quoted:
                depth += (c == "(") - (c == ")")
            i += 1
        yield text[m.end():i - 1]


def missing(text):
    out = []
    for s in asm_statements(text):
        body, _, clobbers = s.rpartition(":")
        out += [(reg, s) for pat, reg in FIXED.items() if re.search(pat, s) and not re.search(f'"{reg}"', clobbers)]
    return out


def test_the_check_sees_a_missing_clobber():
    assert missing('asm volatile("s_mov_b32 m0, %0" ::"s"(f(x)) : "memory");')
    assert not missing('asm volatile("s_mov_b32 m0, %0" ::"s"(f(x)) : "memory", "m0");')


def test_fixed_registers_are_named_as_clobbered():
    files = sorted(glob.glob(os.path.join(PKG, "csrc", "*.h*")))
    found = {os.path.basename(f): missing(open(f).read()) for f in files}
    assert files and not {f: m for f, m in found.items() if m}
