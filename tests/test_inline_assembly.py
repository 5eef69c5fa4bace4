"""Inline assembly says what it changes (the sources' text, no GPU)."""

import re

from tensorfold_amd import build

SOURCES = {p.name: p.read_text() for p in sorted(build.CSRC.iterdir()) if p.suffix in (".hip", ".h")}


def statements(register):
    """(file, text) of the asm statements that move a value to ``register``."""

    return [(name, m[0]) for name, text in SOURCES.items()
            for m in re.finditer(r"asm volatile\(.*?\)(;|\n)", text, re.S) if re.search(rf"s_mov_b32 {register}\b", m[0])]


def test_a_statement_that_writes_m0_declares_it():
    found = statements("m0")
    assert found
    for name, text in found:
        assert '"m0"' in text.rsplit(":", 1)[1], (name, text)


def test_a_scalar_base_may_come_from_a_vector_instruction():
    """Five wait states from a vector instruction's write of a scalar register to a vector memory instruction that reads
    it: the bases of the loads to LDS pass an ``s_nop 3``, and each load begins with the move to m0."""

    text = SOURCES["decode.hip"]
    settled = re.search(r"void settled\(.*?asm volatile\(\"s_nop (\d+)\" : \"\+s\"\(a\), \"\+s\"\(b\), \"\+s\"\(c\)\)", text, re.S)
    assert settled and int(settled[1]) + 1 + 1 >= 5
    request = text[text.index("auto request = "):]
    request = request[:request.index("};")]
    bases = re.search(r"settled\((\w+), (\w+), (\w+)\);", request)
    assert bases
    loads = re.findall(r"[^_]to_lds\d+\((\w+)", request[bases.end():])
    assert len(loads) == 3 and set(loads) == set(bases.groups())
    assert not re.search(r"to_lds\d+\(", request[:bases.start()])
