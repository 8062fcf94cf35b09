"""Inline assembly says which registers it writes by name: what it leaves out the compiler takes as unchanged."""

import re
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "socrates_amd" / "csrc"
SOURCES = sorted(p for p in CSRC.iterdir() if p.suffix in (".hip", ".h"))


def blocks(text):
    """The arguments of every asm statement, comments taken out."""
    text = re.sub(r"//[^\n]*", "", text)
    for found in re.finditer(r"\basm\s+(?:volatile\s*)?\(", text):
        depth, i, quoted = 1, found.end(), False
        while depth:
            c = text[i]
            if c == '"' and text[i - 1] != "\\":
                quoted = not quoted
            elif not quoted:
                depth += (c == "(") - (c == ")")
            i += 1
        yield text[found.end():i - 1]


def named_writes(block):
    code = block.split('" :')[0].split('" ::')[0].split('"\n')[0]
    return {m.group(1) for m in re.finditer(r"\b[sv]_\w+\s+(m0|vcc|exec|scc|[sv]\d+|[sv]\[\d+:\d+\])\b", code)}


@pytest.mark.parametrize("source", SOURCES, ids=lambda p: p.name)
def test_written_registers_are_clobbers(source):
    for block in blocks(source.read_text()):
        for register in named_writes(block):
            assert f'"{register}"' in block, f"{source.name}: {block}"


def test_the_search_finds_such_a_write():
    good, bad = (f'asm volatile("s_mov_b32 m0, %0\\n\\ts_nop 0" ::"s"(x) : {c}); g(1);' for c in ('"memory", "m0"', '"memory"'))
    assert [named_writes(b) for t in (good, bad) for b in blocks(t)] == [{"m0"}, {"m0"}]
    assert '"m0"' in next(blocks(good)) and '"m0"' not in next(blocks(bad))
