#!/usr/bin/env python3
"""Writes rows29_columns.inc: the wave-uniform constant product of fr29.hpp
(rows29) as one inline-asm block per column, and the column blocks that add a
second product to mont29's (dual29).

Column k (0..8) adds x_i * W_{i,k} for i = 0..8, the column's words w[i] held
in SGPRs, and columns 1..7 + D subtract the D Montgomery digits' multiples of r
(m_d * (-r_{k-d}), 1 <= k - d <= 8) in the same signed 64-bit accumulator: a
chain of v_mad_i64_i32 whose carry-out lane masks are discarded (bounds in
fr29.hpp).  Block k first closes column k - 1 into a new accumulator by an
arithmetic shift right by 29, after adding 2^28 when RND says that the
previous column's digit was taken balanced; the previous accumulator stays
intact for that digit.  Block 7 + D is the last that adds terms; block 8 + D
only closes it.

Mac29Col<k> adds x_i * w_{k-i} (both per lane) to the accumulator of column k.

    python3 gen_rows29_columns.py > rows29_columns.inc
"""


def terms(k, d):
    """[(x, y)] of column k with d Montgomery digits."""
    out = [("x[%d]" % i, "w[%d]" % i) for i in range(9)] if k <= 8 else []
    for j in range(d):
        if 1 <= k - j <= 8:
            out.append(("m[%d]" % j, "nr29(%d)" % (k - j)))
    return out


def block(k, d, rnd):
    """(asm text, input operand list).  Operands: %0 the new accumulator, %1 a
    discarded carry mask, %2 the previous column's accumulator (k >= 1),
    [%3 the constant 2^28 (rnd)], then the product pairs."""
    lines, ins, nxt = [], [], 2
    if k >= 1:
        ins.append('"v"(prev)')
        if rnd:
            ins.append('"s"(1u << 28)')
            lines.append("v_mad_i64_i32 %%0, %%1, 1, %%%d, %%%d" % (nxt + 1, nxt))
            lines.append("v_ashrrev_i64 %0, 29, %0")
            nxt += 2
        else:
            lines.append("v_ashrrev_i64 %%0, 29, %%%d" % nxt)
            nxt += 1
    for j, (x, y) in enumerate(terms(k, d)):
        lines.append("v_mad_i64_i32 %%0, %%1, %%%d, %%%d, %s" % (nxt, nxt + 1, "0" if k == 0 and j == 0 else "%0"))
        ins += ['"v"(%s)' % x, '"s"(%s)' % y]
        nxt += 2
    return "\\n\\t".join(lines), ins


def emit(k, d, rnd):
    text, ins = block(k, d, rnd)
    print("template <> struct Rows29Col<%d, %d, %s> {" % (k, d, "true" if rnd else "false"))
    print("  __device__ __forceinline__ static void run(uint64_t& acc, uint64_t prev, const uint32_t* x,")
    print("                                             const uint32_t* w, const uint32_t* m) {")
    print("    uint64_t d;")
    print('    asm("%s"' % text)
    print('        : "=&v"(acc), "=&s"(d)')
    print("        : %s);" % ", ".join(ins))
    print("    (void)d; (void)prev; (void)x; (void)w; (void)m;")
    print("  }")
    print("};")


def emit_mac(k):
    lines, ins, nxt = [], [], 2
    for i in range(max(0, k - 8), min(k, 8) + 1):
        lines.append("v_mad_i64_i32 %%0, %%1, %%%d, %%%d, %%0" % (nxt, nxt + 1))
        ins += ['"v"(x[%d])' % i, '"v"(w[%d])' % (k - i)]
        nxt += 2
    print("template <> struct Mac29Col<%d> {" % k)
    print("  __device__ __forceinline__ static void run(uint64_t& acc, const uint32_t* x, const uint32_t* w) {")
    print("    uint64_t d;")
    print('    asm("%s"' % "\\n\\t".join(lines))
    print('        : "+v"(acc), "=&s"(d)')
    print("        : %s);" % ", ".join(ins))
    print("    (void)d;")
    print("  }")
    print("};")


def main():
    print("// Generated by gen_rows29_columns.py: one asm block per column of the")
    print("// wave-uniform constant product in fr29.hpp (see that script).")
    print("template <int K, int D, bool RND> struct Rows29Col;")
    for d in (1, 2):
        for rnd in (False, True):
            # only the output columns (digit k - 1 >= d) can be balanced
            for k in range(d + 1 if rnd else 0, 9 + d):
                emit(k, d, rnd)
    print("template <int K> struct Mac29Col;")
    for k in range(17):
        emit_mac(k)


if __name__ == "__main__":
    main()
