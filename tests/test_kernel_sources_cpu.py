"""What the kernels' inline assembly may say, read from the sources: the compiler has to know everything it could break."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(__file__), "..", "ksearch_amd", "csrc")


def statements():
    """(file, template, rest) of every asm statement: its instructions and what stands behind them."""
    out = []
    for f in sorted(os.listdir(CSRC)):
        if not f.endswith((".hip", ".hpp", ".cpp")):
            continue
        text = open(os.path.join(CSRC, f)).read()
        for m in re.finditer(r"\basm\b(?:\s+volatile)?\s*\(", text):
            depth, at, quoted = 1, m.end(), False
            while depth:
                c = text[at]
                if c == '"' and text[at - 1] != "\\":
                    quoted = not quoted
                elif not quoted:
                    depth += (c == "(") - (c == ")")
                at += 1
            body = text[m.end():at - 1]
            template = re.match(r'\s*((?:"(?:[^"\\]|\\.)*"\s*)+)', body).group(1)
            out.append((f, template, body[len(template):] if body.startswith(template) else body.split(template, 1)[1]))
    return out


def test_statements_are_found():
    files = {f for f, _, _ in statements()}
    assert {"ksh_device.hpp", "q4k_mm_rows.hpp", "sdpa_prompt.hpp"} <= files


# A register that an asm statement asks memory or LDS for is filled some time after the statement.  The compiler takes it as filled
# there, so a copy or a spill of it in front of the wait keeps what was in it before.
LOADS = re.compile(r"\b(?:ds_(?:read|load|bpermute|permute|swizzle)|(?:global|buffer|flat|scratch|s)_(?:load|read))\w*")


@pytest.mark.parametrize("file,template,rest", statements())
def test_no_asm_returns_a_value_that_is_on_its_way(file, template, rest):
    outputs = rest.split(":")[1] if ":" in rest else ""
    if LOADS.search(template):
        assert "=" not in outputs and "+" not in outputs, f"{file}: {template}"


# Registers with a name of their own: the compiler has to know what a statement writes there, and what it reads (a request straight
# into LDS reads its place there from m0).
WRITES = re.compile(r"\b[sv]_\w+\s+(m0|vcc|exec|scc)\b")


@pytest.mark.parametrize("file,template,rest", statements())
def test_asm_names_the_registers_it_uses(file, template, rest):
    parts = rest.split(":")
    for reg in WRITES.findall(template):
        assert len(parts) > 3 and f'"{reg}"' in parts[3], f"{file}: {reg} in {template}"
    if re.search(r"_load_lds_|_load_\w+ .*\blds\b", template):
        assert '"{m0}"' in rest, f"{file}: {template}"
