"""What the kernels' inline assembly may say, read from the sources: the compiler has to know everything it could break.  And what
the compiler made of the kernels that sit at the edge of the register file, read from the built library's metadata."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from ksearch_amd import _build

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
            rest = body.split(template, 1)[1]
            out.append((f, template.replace("\\n", "\n").replace("\\t", " "), rest))
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


# A scalar register that a vector instruction has written (the compiler may put a uniform address there by v_readfirstlane) must not
# be read by a vector-memory instruction within five wait states, which the compiler does not count into a statement; scalar
# instructions wait for such a register by themselves.  So an address in scalar registers goes through one in the statement.
VECTOR_MEMORY = re.compile(r"\b(?:global|buffer|flat|scratch)_(?:load|store|atomic)[^\n]*")


@pytest.mark.parametrize("file,template,rest", statements())
def test_asm_requests_take_no_scalar_address_as_it_comes(file, template, rest):
    operands = re.findall(r'"([^"]*)"\s*\(', rest)
    for request in VECTOR_MEMORY.findall(template):
        for n in re.findall(r"%(\d+)", request):
            assert operands[int(n)].strip("=&+") != "s", f"{file}: {request}"


def kernels():
    """{kernel: its metadata} of every gfx950 code object in the built library."""
    msgpack = pytest.importorskip("msgpack")
    lib, magic, out, at = open(_build.LIB_PATH, "rb").read(), b"__CLANG_OFFLOAD_BUNDLE__", {}, 0
    while (at := lib.find(magic, at)) >= 0:
        n, = struct.unpack_from("<Q", lib, at + 24)
        entry = at + 32
        for _ in range(n):
            offset, size, id_len = struct.unpack_from("<QQQ", lib, entry)
            name = lib[entry + 24:entry + 24 + id_len]
            entry += 24 + id_len
            if not size or _build.ARCH.encode() not in name:
                continue
            elf = lib[at + offset:at + offset + size]
            table, = struct.unpack_from("<Q", elf, 0x28)
            each, sections = struct.unpack_from("<HH", elf, 0x3A)
            for i in range(sections):
                kind, place = struct.unpack_from("<4xI16xQ", elf, table + i * each)
                if kind != 7:                                  # SHT_NOTE
                    continue
                owner, length, note = struct.unpack_from("<III", elf, place)
                if note == 32:                                 # NT_AMDGPU_METADATA
                    begin = place + 12 + (owner + 3) // 4 * 4
                    for k in msgpack.unpackb(elf[begin:begin + length])["amdhsa.kernels"]:
                        out[k[".name"]] = k
        at += len(magic)
    return out


# Kernels that fill their registers to fit two (or four) workgroups on a compute unit, and wait by the number of their requests: what
# goes to memory and back beside those makes every such wait longer.
FULL = re.compile(r"q[46]k_mm_rows_kernel|sdpa_prompt_kernel|q4k_mm_round_kernel|q4k_mm_skinny_kernel")


def test_full_kernels_keep_their_values_in_registers():
    found = {name: k for name, k in kernels().items() if FULL.search(name)}
    assert len(found) >= 18
    spilled = {name: (k[".vgpr_spill_count"], k[".private_segment_fixed_size"]) for name, k in found.items()
               if k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]}
    assert not spilled


@pytest.mark.skipif(not shutil.which("hipcc"), reason="needs the compiler")
@pytest.mark.parametrize("shape,taken", [("2, 2, 1, 4", True), ("1, 2, 1, 4", True), ("1, 1, 1, 4", True), ("4, 1, 1, 4, false", True), ("2, 1, 1, 4, false", True),
                                         ("1, 1, 2, 2", True), ("2, 1, 2, 2, false", False), ("3, 1, 1, 4, false", False)])
def test_prompt_gemm_takes_only_shapes_that_its_waits_count(shape, taken):
    """q4k_mm_rows_kernel waits by the number of its requests, which its units issue at places fixed at compile time: a shape with
    fewer places than requests would read LDS ahead of what it waits for, so it does not compile.  (Four token tiles, or three, to
    waves that have two places for a superblock's sums.)"""
    r = subprocess.run(["hipcc", "-x", "hip", "-std=c++17", f"--offload-arch={_build.ARCH}", "--offload-host-only", "-fsyntax-only", "-w", "-I" + CSRC, "-"],
                       input=f'#include "mul_mm_q4k.hip"\nstatic_assert(ksh::MmRows<{shape}>::TM > 0, "");\n', capture_output=True, text=True)
    assert (r.returncode == 0) == taken, r.stderr[-500:]
    assert taken or "static assertion failed" in r.stderr
