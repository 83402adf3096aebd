"""Generates nt_math_tables.h: constants of the skeleton's own fp64 math.

* log (Tang's table-driven method, ACM TOMS 16(4), 1990), producing -2 ln u
  for Box-Muller: the argument is scaled to x in about [3/4, 3/2) and F is x
  rounded to 8 fractional bits of its binade, F = from_hi(0x3FE80000 + (j <<
  12)), j = 0..255 (F = 1 at j = 128). The table holds i' = -2 i with i the
  double nearest 1/F, so that r' = -2 (x i - 1) is one fma, exact to a
  rounding, and 2 ln i as head + tail (heads on a 2^-42 grid, -2 ln 2's head
  with 42 bits, so e (-2 ln2_hi) + head is exact). ln(1 + r), |r| <= 2^-9, is
  the Taylor polynomial through r^6 (truncation below r^6/7 < 1e-17 relative),
  rewritten in r' = -2 r.
* exp (Tang's table-driven method, ACM TOMS 15(2), 1989): x = (256 m + j)
  ln2/256 + r, |r| <= ln2/512; the table holds 2^(j/256) as head and tail;
  ln2/256 is split into a head with 32 significant bits and a tail; exp(r) - 1
  is the Taylor polynomial through r^4.
* sin / cos on the full circle: the angle's sector j (of 512) has a table
  angle a_j near its middle, a multiple of 2^-40 chosen so that sin a_j and cos
  a_j are doubles to within a few hundredths of an ulp (accurate tables: Gal
  and Bachelis, ACM TOMS 17(1), 1991), and those two; w = theta - a_j, |w| <=
  pi/512 + 2^-28, sin w through w^5 (Taylor, truncation below
  7e-20) and cos w - 1 through w^4 (Taylor, with the w^4 coefficient moved to
  level the error: below 1e-17).
* the tables and coefficients of the routines that reduce in turns: -2/F and
  -2 ln F for F = x to 8 fractional bits in [sqrt(1/2), sqrt(2)), (sin, cos)(2
  pi j / 512), sin and cos polynomials in turns.
* ln 2 as a double-double; the reference's 2 pi literal.
All values are computed here with mpmath at 60 digits and rounded once.
Run: python nablatensor_amd/csrc/gen_math_tables.py
"""
from __future__ import annotations

import struct
from pathlib import Path

import mpmath as mp
import numpy as np

mp.mp.dps = 60


def hexd(x: float) -> str:
    return float(x).hex()


def from_hi(hi: int) -> float:
    return struct.unpack("<d", struct.pack("<Q", hi << 32))[0]


def main() -> None:
    lines = ["// generated by gen_math_tables.py (mpmath, 60 digits); do not edit", "#pragma once", ""]
    # Heads are multiples of 2^-43 and ln2_hi has 42 significant bits, so
    # e * ln2_hi + head is exact for |e| < 2^10 (Tang's exact-head layout).
    def head(v, ulp_exp):
        q = mp.mpf(2) ** ulp_exp
        return float(mp.nint(v / q) * q)

    def arr(vals):
        return ",\n    ".join(", ".join(hexd(v) for v in vals[i:i + 4]) for i in range(0, len(vals), 4))

    # Every log entry is stored times -2 (exact), so the kernel gets -2 ln u
    # without a final multiply: the same bits as -2 * (Tang's ln u).
    inv, lo_hi, lo_lo = [], [], []
    for idx in range(256):
        F = from_hi(0x3FE80000 + (idx << 12))
        i = float(mp.mpf(1) / mp.mpf(F))
        inv.append(-2.0 * i)
        l = -mp.log(mp.mpf(i))
        h = head(l, -43)
        lo_hi.append(-2.0 * h)
        lo_lo.append(-2.0 * float(l - mp.mpf(h)))
    assert inv[128] == -2.0 and lo_hi[128] == 0.0 and lo_lo[128] == 0.0
    ln2 = mp.log(2)
    ln2_hi = head(ln2, -42)
    ln2_lo = float(ln2 - mp.mpf(ln2_hi))
    lines.append(f"#define NT_M2LN2_HI {hexd(-2.0 * ln2_hi)}  /* -2 ln 2, 42-bit head */")
    lines.append(f"#define NT_M2LN2_LO {hexd(-2.0 * ln2_lo)}")
    # -2 ln(1 + r) = r' + r'^2 Q(r'), r' = -2 r, Q_k = -(1/2)(-1/2)^k c_k for
    # ln(1 + r) = r + r^2 (c_0 + c_1 r + ...), c_k = (-1)^(k+1) / (k + 2)
    for k in range(5):
        c = mp.mpf((-1) ** (k + 1)) / (k + 2)
        qk = float(c) * (-0.5) * (-0.5) ** k
        assert qk == float(c * mp.mpf(-0.5) * mp.mpf(-0.5) ** k)
        lines.append(f"#define NT_LOGQ_{k} {hexd(qk)}")
    tp = 2 * mp.pi
    two_pi_d = 6.283185307179586  # the reference's literal for 2 pi (Philox.java:74)
    lines.append(f"#define NT_TWO_PI_D {hexd(two_pi_d)}")
    lines.append(f"#define NT_TWO_PI_U32 {hexd(two_pi_d * 2.0 ** -32)}  /* NT_TWO_PI_D 2^-32, exact */")
    # exp: 2^(j/256) head + tail, ln2/256 = L_hi (32 significant bits) + L_lo
    l64 = ln2 / 256
    e = mp.floor(mp.log(l64, 2))
    q = mp.mpf(2) ** (e - 31)
    l_hi = float(mp.nint(l64 / q) * q)
    l_lo = float(l64 - mp.mpf(l_hi))
    lines.append(f"#define NT_EXP_INV_L {hexd(float(256 / ln2))}  /* 256 / ln 2 */")
    lines.append(f"#define NT_EXP_L_HI {hexd(l_hi)}  /* ln2/256, 32-bit head */")
    lines.append(f"#define NT_EXP_L_LO {hexd(l_lo)}")
    for k in range(2, 5):
        lines.append(f"#define NT_EXP_C{k} {hexd(float(mp.mpf(1) / mp.factorial(k)))}")
    exp_h, exp_l = [], []
    for j in range(256):
        v = mp.mpf(2) ** (mp.mpf(j) / 256)
        h = float(v)
        exp_h.append(h)
        exp_l.append(float(v - mp.mpf(h)))

    def struct(name, init, fields):
        lines.append("")
        lines.append("struct __attribute__((aligned(16))) " + name + " {")
        for f, vals, note in fields:
            pad = 1 if len(fields) > 1 else 0
            lines.append(f"  double {f}[{len(vals) + pad}];  /* {note} */")
        lines.append("};")
        lines.append(f"#define {init} {{ \\")
        lines.append(", \\\n".join("  {" + arr(vals).replace("\n", " \\\n") + "}" for _, vals, _ in fields) + " }")

    def pairs(a, b):
        return [v for ab in zip(a, b) for v in ab]

    struct("NtExpTable", "NT_EXP_TABLE_INIT", [("t", pairs(exp_h, exp_l), "t[2j] + t[2j+1] = 2^(j/256)")])
    # sin w = w + w t (S3 + S5 t), cos w - 1 = t (-1/2 + C4 t), t = w^2
    for k in (3, 5):
        lines.append(f"#define NT_SC_S{k} {hexd(float(mp.mpf((-1) ** (k // 2)) / mp.factorial(k)))}")
    # t <= T = (pi/512)^2: C4 also takes the w^6 term's share that minimises
    # the largest error on [0, T]. The error left is t^2 (delta - c6 t) with
    # delta = C4' - C4 and c6 the w^6 Taylor coefficient; delta = beta c6 T
    # with 4 beta^3 / 27 = 1 - beta levels the interior extremum (at t = 2
    # beta T / 3) with the end point t = T, a tenth of the plain truncation.
    c6 = -mp.mpf(1) / mp.factorial(6)
    beta = mp.findroot(lambda b: 4 * b ** 3 / 27 - (1 - b), 0.9)
    lines.append(f"#define NT_SC_C4 {hexd(float(mp.mpf(1) / 24 + beta * c6 * (mp.pi / 512) ** 2))}")
    ang, sn, cs = [], [], []
    for j in range(512):
        a = float(mp.nint(tp * (j + mp.mpf(1) / 2) / 512 * 2 ** 40) / mp.mpf(2) ** 40)
        # of the 8,193 multiples of 2^-40 around it, the angle whose sine and
        # cosine both lie closest to doubles (searched in long double)
        near = (a + np.arange(-4096, 4097) * 2.0 ** -40).astype(np.longdouble)
        off = np.maximum(*(np.abs(v - v.astype(np.float64)) / np.spacing(np.abs(v.astype(np.float64)))
                           for v in (np.sin(near), np.cos(near))))
        a = float(near[np.argmin(off)])
        ang.append(a)
        sn.append(float(mp.sin(mp.mpf(a))))
        cs.append(float(mp.cos(mp.mpf(a))))
    struct("NtSinCosTable", "NT_SINCOS_TABLE_INIT",
           [("sin", sn, "sin a_j"), ("cos", cs, "cos a_j"), ("ang", ang, "a_j, near 2 pi (j + 1/2) / 512")])
    struct("NtLogTable", "NT_LOG_TABLE_INIT",
           [("inv", inv, "-2 i, i = 1/F rounded"), ("hi", lo_hi, "2 ln i, head"), ("lo", lo_lo, "tail")])
    # the tables of the routines that reduce in turns (NT_TURN_DRAWS)
    inv, lo_hi, lo_lo = [], [], []
    for idx in range(257):
        F = from_hi(0x3FE6A000 + (idx << 12))
        inv.append(-2.0 * float(mp.mpf(1) / mp.mpf(F)))
        l = mp.log(mp.mpf(F))
        h = head(l, -43)
        lo_hi.append(-2.0 * h)
        lo_lo.append(-2.0 * float(l - mp.mpf(h)))
    assert from_hi(0x3FE6A000 + (150 << 12)) == 1.0 and lo_hi[150] == 0.0
    lines.append(f"#define NT_TWO_PI_D_ERR {hexd(float(mp.mpf(two_pi_d) - tp))}  /* NT_TWO_PI_D - 2 pi */")
    for k in (1, 3, 5):
        lines.append(f"#define NT_TURN_S{k} {hexd(float((-1) ** (k // 2) * tp ** k / mp.factorial(k)))}")
    c6 = -(tp ** 6) / mp.factorial(6)  # the f^4 coefficient levelled as C4 above, on |f| <= 2^-10 turns
    turn_c = {2: -(tp ** 2) / 2, 4: tp ** 4 / 24 + beta * c6 * mp.mpf(2) ** -20}
    for k in (2, 4):
        lines.append(f"#define NT_TURN_C{k} {hexd(float(turn_c[k]))}")
    sn = [float(mp.sin(tp * j / 512)) for j in range(512)]
    cs = [float(mp.cos(tp * j / 512)) for j in range(512)]
    struct("NtTurnTable", "NT_TURN_TABLE_INIT", [("t", pairs(sn, cs), "t[2j], t[2j+1] = sin, cos of 2 pi j / 512")])
    struct("NtTurnLogTable", "NT_TURN_LOG_TABLE_INIT",
           [("inv", inv, "-2 / F"), ("hi", lo_hi, "-2 ln F, head"), ("lo", lo_lo, "tail")])
    lines.append("")
    lines.append("// All tables in one LDS block. Columns that share an index are arrays of their own")
    lines.append("// (one address for all of them), one entry longer than they need: at a distance that")
    lines.append("// is a multiple of 512 bytes two reads become one ds_read2st64_b64, which kept the")
    lines.append("// LDS busy 1.4 times as long (SQ_LDS_IDX_ACTIVE of the 252-step Asian kernel on 2x10^6")
    lines.append("// paths: 2.90e8 against 2.06e8, with a quarter fewer instructions).")
    lines.append("#ifdef NT_TURN_DRAWS")
    lines.append("struct __attribute__((aligned(16))) NtTables {\n  NtTurnTable sc;\n  NtExpTable ex;\n  NtTurnLogTable lg;\n};")
    lines.append("#define NT_TABLES_INIT { NT_TURN_TABLE_INIT, NT_EXP_TABLE_INIT, NT_TURN_LOG_TABLE_INIT }")
    lines.append("#else")
    lines.append("struct __attribute__((aligned(16))) NtTables {\n  NtSinCosTable sc;\n  NtExpTable ex;\n  NtLogTable lg;\n};")
    lines.append("#define NT_TABLES_INIT { NT_SINCOS_TABLE_INIT, NT_EXP_TABLE_INIT, NT_LOG_TABLE_INIT }")
    lines.append("#endif")
    out = Path(__file__).resolve().parent / "nt_math_tables.h"
    out.write_text("\n".join(lines) + "\n")
    print("wrote", out)


if __name__ == "__main__":
    main()
