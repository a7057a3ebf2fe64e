"""Writes mcdp_log_table.hpp: the table of the samplers' logarithm (log_tab in mcdp_math.hpp).

With hx the high word of x, kLogBase - hx = 2^20 m + 2^12 j + (low bits) names a scale and an interval:
z = x 2^m lies in interval j of 256, whose middle c_j is the double of high word
kLogBase + 1 - 2^11 - 2^12 j and low word 0 (c from 1.375 down to 0.69; 1.0 is one of them).  For each
interval: inv_j = 1/c_j rounded to a multiple of 2^-10 (so that z inv_j - 1 needs hardly more than a double's
53 bits and its rounding all but vanishes), and -log(inv_j) split as hi + lo, hi the multiple of 2^-32
nearest it (so hi - m ln2_hi is exact for every binary exponent), lo the rest rounded to double.  Values
come from the host's 80-bit long double logarithm (64-bit significand); hi + lo is within 2^-64 of
-log(inv_j).

Run: python mc_dagprop_amd/csrc/gen_log_table.py  (rewrites the header next to this file).
"""

from __future__ import annotations

import pathlib

import numpy as np

N = 256
BASE = 0x3FF00000 + 0x60000 + 0x800 - 1  # the largest high word of z: 1.375 + half an interval


def table() -> tuple[list[float], list[float], list[float]]:
    LD = np.longdouble
    assert np.finfo(LD).nmant >= 63, "needs x87 long double"
    inv, hi, lo = [], [], []
    for j in range(N):
        word = BASE + 1 - 0x800 - 0x1000 * j
        c = float(np.array([word << 32], dtype=np.uint64).view(np.float64)[0])
        v = float(np.rint(1024.0 / c)) / 1024.0
        lf = -np.log(LD(v))
        h = float(np.rint(lf * LD(2.0**32)) / LD(2.0**32))
        assert h == np.ldexp(np.rint(np.ldexp(h, 32)), -32)
        inv.append(v)
        hi.append(h)
        lo.append(float(lf - LD(h)))
    assert any(v == 1.0 and h == 0.0 and l == 0.0 for v, h, l in zip(inv, hi, lo))
    return inv, hi, lo


def render() -> str:
    inv, hi, lo = table()

    def arr(name: str, vals: list[float], size: str, per_line: int) -> str:
        body = ",\n".join("    " + ", ".join(float.hex(v) for v in vals[i:i + per_line])
                          for i in range(0, len(vals), per_line))
        return f"__device__ __attribute__((aligned(16))) const double {name}[{size}] = {{\n{body}}};\n"

    hilo = [v for pair in zip(hi, lo) for v in pair]
    return (
        "// Generated by gen_log_table.py: the intervals of log_tab (mcdp_math.hpp).  kLogInv[j] = 1/c_j rounded to\n"
        "// 2^-10; -log(kLogInv[j]) = kLogHiLo[2j] + kLogHiLo[2j + 1], the first a multiple of 2^-32.\n"
        "#pragma once\n#include <hip/hip_runtime.h>\n\nnamespace mcdp {\n\n"
        f"constexpr int kLogTableSize = {N};\nconstexpr uint32_t kLogBase = 0x{BASE:08x}u;\n\n"
        + arr("kLogInv", inv, "kLogTableSize", 4) + "\n" + arr("kLogHiLo", hilo, "2 * kLogTableSize", 4)
        + "\n}  // namespace mcdp\n"
    )


if __name__ == "__main__":
    out = pathlib.Path(__file__).resolve().parent / "mcdp_log_table.hpp"
    out.write_text(render())
    print(f"wrote {out}")
