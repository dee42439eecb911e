"""Generate adana_pow_tables.h: the lookup tables of the binary64 pow core.

log table (128 entries, j = top 7 mantissa bits of x in [1, 2)), stored as
16-byte pairs {inv_c, neg_log2} so that one 16-byte load fetches both:
  inv_c[j]  ~ 1 / (1 + (j + 0.5) / 128) rounded to 12 significant bits, so
            that m * inv_c[j] is exact in binary64 for a 24-bit m;
  neg_log2[j] = -log2(inv_c[j]) in binary64 (computed with 60-digit decimals).
exp table (128 entries): two_j[j] = 2^(j/128) in binary64.
Run:  python adana_amd/csrc/gen_pow_tables.py > adana_amd/csrc/adana_pow_tables.h
"""
from decimal import Decimal, getcontext
import math

getcontext().prec = 60
LN2 = Decimal(2).ln()


def round_sig(x: float, bits: int) -> float:
    m, e = math.frexp(x)
    return math.ldexp(round(m * (1 << bits)) / (1 << bits), e)


def dec_ln(x: float) -> Decimal:
    return Decimal(x).ln()


def main():
    out = ["// Generated by gen_pow_tables.py -- do not edit.",
           "#ifndef ADANA_POW_TABLES_H", "#define ADANA_POW_TABLES_H", "",
           "namespace adana {", ""]
    inv = [round_sig(1.0 / (1.0 + (j + 0.5) / 128.0), 12) for j in range(128)]
    negl = [float(-dec_ln(v) / LN2) for v in inv]
    two = [float((LN2 * Decimal(j) / Decimal(128)).exp()) for j in range(128)]
    def fmt(vals, name):
        # 16-byte aligned: the step kernel copies it to LDS in 16-byte words
        lines = [f"alignas(16) ADANA_TABLE_ATTR const double {name}[128] = {{"]
        for i in range(0, 128, 4):
            lines.append("    " + ", ".join(v.hex() for v in vals[i:i + 4]) + ",")
        lines.append("};")
        return lines
    out += ["struct alignas(16) LogPair {", "    double inv_c, neg_log2;", "};", "",
            "ADANA_TABLE_ATTR const LogPair kLog[128] = {"]
    out += [f"    {{{a.hex()}, {b.hex()}}}," for a, b in zip(inv, negl)]
    out += ["};", ""] + fmt(two, "kExp2J") + [""]
    out += ["}  // namespace adana", "", "#endif  // ADANA_POW_TABLES_H", ""]
    print("\n".join(out))


if __name__ == "__main__":
    main()
