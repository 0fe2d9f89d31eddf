"""Accumulators that pass between matrix products of different shapes, in the
built library's gfx950 code (no device needed).

The compiler leaves no wait where a product continues the accumulator of a
product of another shape, as it needs none between products of one shape.  The
sources wait there themselves, 8 states as for a vector instruction that reads
a product's result: every such pair in the code must be that far apart.
"""
import re
import shutil
import struct
import subprocess

import pytest

from stepquant_amd import _native as N

OBJDUMP = shutil.which("llvm-objdump", path="/opt/rocm/llvm/bin")
WAIT = 8


def _code_object(data):
    """The gfx950 ELF of the library's offload bundle."""
    at = data.index(b"__CLANG_OFFLOAD_BUNDLE__")
    n, = struct.unpack_from("<Q", data, at + 24)
    pos = at + 32
    for _ in range(n):
        offset, size, length = struct.unpack_from("<QQQ", data, pos)
        name = data[pos + 24:pos + 24 + length]
        pos += 24 + length
        if name.endswith(b"gfx950"):
            return data[at + offset:at + offset + size]
    raise AssertionError("no gfx950 code in the library")


def _registers(operand):
    m = re.match(r"v\[(\d+):(\d+)\]", operand)
    return set(range(int(m[1]), int(m[2]) + 1)) if m else set()


def close_pairs(listing):
    """(kernel, wait states, first product, second) of the pairs nearer than
    WAIT, along straight code (jumps only add to a distance)."""
    found, kernel, open_products, products = [], "", [], 0
    for line in listing:
        if line.endswith(">:"):
            kernel, open_products = line.split("<")[-1][:-2], []
            continue
        text = line.split("//")[0].strip()
        op, _, rest = text.partition(" ")
        if not op:
            continue
        states = int(rest, 0) + 1 if op == "s_nop" else 1
        if op.startswith("v_mfma"):
            products += 1
            operands = [x.strip() for x in re.split(r",(?![^\[]*\])", rest)]
            wrote, accumulator = _registers(operands[0]), _registers(operands[3])
            found += [(kernel, age, first, text) for age, shape, regs, first in open_products
                      if shape != op and regs & accumulator]
            # a register that is written again belongs to the newer product
            open_products = [(a, s, r - wrote, t) for a, s, r, t in open_products]
        open_products = [(a + states, s, r, t) for a, s, r, t in open_products if r and a + states < WAIT]
        if op.startswith("v_mfma"):
            open_products.append((0, op, wrote, text))
    return found, products


def test_close_pairs_are_found():
    first = "v_mfma_f32_16x16x32_bf16 v[82:85], v[82:85], v[90:93], v[98:101]"
    second = "v_mfma_f32_16x16x16_bf16 v[82:85], v[86:87], v[116:117], v[82:85]"
    other = "v_and_b32_e32 v90, 0xffff0000, v117"
    assert len(close_pairs(["<k>:", first, other, second])[0]) == 1
    assert len(close_pairs(["<k>:", first, "s_nop 6", second])[0]) == 1
    assert not close_pairs(["<k>:", first, "s_nop 7", second])[0]
    assert not close_pairs(["<k>:", first, first.replace("v[98:101]", "v[82:85]")])[0]  # one shape
    assert not close_pairs(["<k>:", first, second.replace("v[82:85]", "v[70:73]")])[0]


@pytest.mark.skipif(OBJDUMP is None, reason="llvm-objdump is not installed")
def test_accumulators_between_shapes_are_waited_for(tmp_path):
    with open(N.LIB_PATH, "rb") as f:
        elf = _code_object(f.read())
    (tmp_path / "code").write_bytes(elf)
    out = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--mcpu=gfx950", str(tmp_path / "code")], check=True,
                         capture_output=True, text=True).stdout
    found, products = close_pairs(out.splitlines())
    assert products > 1000 and not found
