"""Generate zodi_math_tables.inc: correctly rounded tables for the device exp/log.

* EXP2_TABLE[j] = 2^(j/256), j = 0..255 (table-driven exp, Tang 1989,
  ACM TOMS 15(2):144-157);
* LOG_INV[j] = 1/c_j and LOG_C[j] = log(c_j) with c_j = 1/2 + j/512,
  j = 0..255 (table-driven log, Tang 1990, ACM TOMS 16(4):378-400);
* LINE_INV[j] = 1/(1/2 + (j + 1/2)/512) rounded to a multiple of 2^-12 and
  LINE_LOG[j] = -log(LINE_INV[j]) (zodi_line_math.hpp: the product of a mantissa and a
  13-bit LINE_INV is exact inside an FMA).
* EXP2_LO[j] and LINE_LOG2[2 j], LINE_LOG2[2 j + 1]: what EXP2_TABLE[j] leaves out of
  2^(j/256), and -log2(LINE_INV[j]) in two words (zodi_line_math.hpp: build_pow_table).
* LINE_ANGLE[2 j], LINE_ANGLE[2 j + 1] = cos, sin of the exact product of j and the double
  pi/128, j = 0..128 (zodi_line_math.hpp: unit_angle).

Values are evaluated with mpmath at 200 bits and rounded to nearest double.
Run ``python -m zodipy_amd.csrc.gen_math_tables`` to regenerate.
"""

from __future__ import annotations

import math
from pathlib import Path

import mpmath

OUT = Path(__file__).resolve().parent / "zodi_math_tables.inc"


def _hex(v) -> str:
    return float(v).hex()


def main() -> None:
    mpmath.mp.prec = 200
    exp2 = [mpmath.power(2, mpmath.mpf(j) / 256) for j in range(256)]
    cs = [mpmath.mpf(1) / 2 + mpmath.mpf(j) / 512 for j in range(256)]
    inv = [1 / c for c in cs]
    logc = [mpmath.log(c) for c in cs]
    lines = [
        "// Generated by gen_math_tables.py (mpmath, 200-bit, rounded to nearest double).",
        "// 2^(j/256), j = 0..255",
        "#define ZODI_EXP2_TABLE \\",
    ]
    lines += [f"  {_hex(v)}, \\" for v in exp2]
    lines[-1] = lines[-1].rstrip(" \\").rstrip(",")
    lines += ["// 1/c_j, c_j = 1/2 + j/512, j = 0..255", "#define ZODI_LOG_INV_TABLE \\"]
    lines += [f"  {_hex(v)}, \\" for v in inv]
    lines[-1] = lines[-1].rstrip(" \\").rstrip(",")
    lines += ["// log(c_j)", "#define ZODI_LOG_C_TABLE \\"]
    lines += [f"  {_hex(v)}, \\" for v in logc]
    lines[-1] = lines[-1].rstrip(" \\").rstrip(",")
    short = [mpmath.nint(4096 / (mpmath.mpf(1) / 2 + (mpmath.mpf(j) + mpmath.mpf(1) / 2) / 512))
             / 4096 for j in range(256)]
    lines += ["// 1/(1/2 + (j + 1/2)/512) to 2^-12", "#define ZODI_LINE_INV_TABLE \\"]
    lines += [f"  {_hex(v)}, \\" for v in short]
    lines[-1] = lines[-1].rstrip(" \\").rstrip(",")
    lines += ["// -log of the same", "#define ZODI_LINE_LOG_TABLE \\"]
    lines += [f"  {_hex(-mpmath.log(v))}, \\" for v in short]
    lines[-1] = lines[-1].rstrip(" \\").rstrip(",")
    low = [v - mpmath.mpf(float(v)) for v in exp2]
    lines += ["// 2^(j/256) less its entry above", "#define ZODI_EXP2_LO_TABLE \\"]
    lines += [f"  {_hex(v)}, \\" for v in low]
    lines[-1] = lines[-1].rstrip(" \\").rstrip(",")
    log2 = [-mpmath.log(v, 2) for v in short]
    pairs = [w for v in log2 for w in (float(v), float(v - mpmath.mpf(float(v))))]
    lines += ["// -log2 of the 1/(1/2 + (j + 1/2)/512), two words each",
              "#define ZODI_LINE_LOG2_TABLE \\"]
    lines += [f"  {_hex(v)}, \\" for v in pairs]
    lines[-1] = lines[-1].rstrip(" \\").rstrip(",")
    angle = [f(j * mpmath.mpf(math.pi / 128)) for j in range(129)
             for f in (mpmath.cos, mpmath.sin)]
    lines += ["// cos and sin of j pi/128", "#define ZODI_LINE_ANGLE_TABLE \\"]
    lines += [f"  {_hex(v)}, \\" for v in angle]
    lines[-1] = lines[-1].rstrip(" \\").rstrip(",")
    OUT.write_text("\n".join(lines) + "\n")
    print(OUT)


if __name__ == "__main__":
    main()
