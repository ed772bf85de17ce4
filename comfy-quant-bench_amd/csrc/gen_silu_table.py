"""Generate the silu tables of the SwiGLU prologue: silu(g) = g / (1 + exp(-g)) correctly rounded
to fp32.

Build step of libmq.so (run by build.py into its build directory).

mq_silu_table.h, bf16 gates. For a gate value g with bit pattern b (|b| = b & 0x7fff):
  |b| <  0x3300 (|g| < 2^-25): RN(silu(g)) = g / 2      (the correction g^2/4 is below half an ulp)
  |b| >= 0x4300 (|g| >= 128):   RN(silu(g)) = g for g > 0 and -0.0 for g < 0 (g e^g underflows)
  otherwise:                    table entry ((|b| - 0x3300) + 4096 * sign) of this file.
mq_silu_f16_table.h, fp16 gates: one entry per 16-bit pattern (65536), indexed by the pattern.
Non-finite gates take the value of the formula in IEEE arithmetic: +inf -> +inf, -inf -> NaN
(-inf / inf), NaN -> NaN.
The values are computed with Python's decimal module at 60 significant digits and rounded to the
nearest fp32 (ties to even), so every finite entry is the correctly rounded fp32 silu of its gate.

    python gen_silu_table.py OUT_HEADER [OUT_F16_HEADER]
"""
from __future__ import annotations

import struct
import sys
from decimal import MAX_EMAX, MIN_EMIN, Decimal, getcontext

LO, HI = 0x3300, 0x4300          # |bf16 bits| range covered by the table (exponent fields 102..133)
ENTRIES = HI - LO                # per sign


def _f32_bits(x: float) -> int:
    return struct.unpack("<I", struct.pack("<f", x))[0]


def _f32_from_bits(u: int) -> float:
    return struct.unpack("<f", struct.pack("<I", u))[0]


def round_to_f32(d: Decimal) -> int:
    """Bits of the fp32 nearest to d (ties to even). d is nonzero and within the fp32 range."""
    approx = float(d)                                    # nearest double
    u = _f32_bits(struct.unpack("<f", struct.pack("<f", approx))[0])
    best = None
    for cand in (u - 1, u, u + 1):
        if cand & 0x7f800000 == 0x7f800000:              # skip inf / nan neighbours
            continue
        err = abs(Decimal(_f32_from_bits(cand)) - d)
        key = (err, cand & 1)                            # ties: even mantissa wins
        if best is None or key < best[0]:
            best = (key, cand)
    return best[1]


def silu_f32_bits(b: int) -> int:
    g = Decimal(_f32_from_bits(b << 16))
    s = g / (1 + (-g).exp())
    if s == 0:
        return 0x80000000 if b & 0x8000 else 0
    return round_to_f32(s)


def silu_f16_gate_bits(b: int) -> int:
    """fp32 bits of silu(g) for the fp16 gate with bit pattern b."""
    g = struct.unpack("<e", struct.pack("<H", b))[0]
    if g != g:                                           # NaN gate
        return 0x7FC00000
    if g == float("inf"):
        return 0x7F800000
    if g == float("-inf"):
        return 0x7FC00000
    d = Decimal(g)
    s = d / (1 + (-d).exp())
    if s == 0:
        return 0x80000000 if (b & 0x8000) else 0
    return round_to_f32(s)


def table_f16() -> list[int]:
    ctx = getcontext()
    ctx.prec, ctx.Emax, ctx.Emin = 60, MAX_EMAX, MIN_EMIN
    return [silu_f16_gate_bits(b) for b in range(0x10000)]


def table() -> list[int]:
    ctx = getcontext()
    ctx.prec, ctx.Emax, ctx.Emin = 60, MAX_EMAX, MIN_EMIN
    out = []
    for sign in (0, 0x8000):
        out.extend(silu_f32_bits(sign | t) for t in range(LO, HI))
    return out


def main_f16(path: str) -> None:
    vals = table_f16()
    lines = [
        "// Generated by gen_silu_table.py: fp32 bits of silu(g) = g / (1 + exp(-g)), correctly rounded,",
        "// for every fp16 gate, indexed by its 16-bit pattern.",
        "#pragma once",
        "#include <cstdint>",
        "namespace mq {",
        "__device__ const uint32_t kSiluF16Table[65536] __attribute__((aligned(16))) = {",
    ]
    for i in range(0, len(vals), 8):
        lines.append("    " + ", ".join(f"0x{v:08x}u" for v in vals[i:i + 8]) + ",")
    lines += ["};", "}  // namespace mq", ""]
    with open(path, "w") as f:
        f.write("\n".join(lines))


def main(path: str) -> None:
    vals = table()
    vals = [v for pair in zip(vals[:ENTRIES], vals[ENTRIES:]) for v in pair]   # the signs interleaved
    lines = [
        "// Generated by gen_silu_table.py: fp32 bits of silu(g) = g / (1 + exp(-g)), correctly rounded,",
        f"// for bf16 gates with 0x{LO:04x} <= (bits & 0x7fff) < 0x{HI:04x}; index 2 * (|bits| - 0x{LO:04x}) + sign.",
        "#pragma once",
        "#include <cstdint>",
        "namespace mq {",
        f"constexpr uint32_t kSiluLo = 0x{LO:04x}u, kSiluEntries = {ENTRIES}u;",
        f"__device__ const uint32_t kSiluTable[{2 * ENTRIES}] __attribute__((aligned(16))) = {{",
    ]
    for i in range(0, len(vals), 8):
        lines.append("    " + ", ".join(f"0x{v:08x}u" for v in vals[i:i + 8]) + ",")
    lines += ["};", "}  // namespace mq", ""]
    with open(path, "w") as f:
        f.write("\n".join(lines))


if __name__ == "__main__":
    main(sys.argv[1])
    if len(sys.argv) > 2:
        main_f16(sys.argv[2])
