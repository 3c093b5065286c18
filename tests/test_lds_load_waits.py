"""Loads that go straight to LDS take their address from M0, and the instruction set asks for one wait state between a scalar write of
M0 and such a load.  The compiler keeps to that for its own code but does not look into inline assembly: every statement that
writes M0 has to have the wait itself.  Read off the sources, no kernel runs here."""
import pathlib
import re

import pytest

SOURCES = sorted(p for p in (pathlib.Path(__file__).resolve().parent.parent / "flh_amd" / "csrc").iterdir() if p.suffix in (".h", ".hip"))


def statements(text):
    """The instructions of every inline assembly statement, in order."""
    for body in re.findall(r'\basm(?:\s+volatile)?\s*\(\s*((?:"(?:[^"\\]|\\.)*"\s*)+)', text):
        code = "".join(re.findall(r'"((?:[^"\\]|\\.)*)"', body))
        yield [i.strip() for i in re.split(r"\\n(?:\\t)?|;", code) if i.strip()]


@pytest.mark.parametrize("path", SOURCES, ids=lambda p: p.name)
def test_m0_is_waited_for(path):
    for code in statements(path.read_text()):
        for i, ins in enumerate(code):
            if re.match(r"s_\w+\s+m0\s*,", ins):
                assert i + 1 < len(code) and code[i + 1].startswith("s_nop"), (path.name, code)


def test_the_reader_sees_them():
    assert sum(any(" m0" in i for i in code) for p in SOURCES for code in statements(p.read_text())) >= 8
