"""The wave-uniform constant product of the NTT passes and scans (rows29 in
csrc/fr29.hpp) and the eight-point DFT built on it (csrc/ntt_pass.hpp), on the
host against Python integers."""
import ctypes
import os
import random
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "ppopp26-artifact_amd", "csrc")
R = 0x73EDA753299D7D483339D80809A1D80553BDA402FFFE5BFEFFFFFFFF00000001
U = ctypes.c_uint32


@pytest.fixture(scope="module")
def rows(tmp_path_factory):
    d = tmp_path_factory.mktemp("rows29")
    src = d / "r.cpp"
    src.write_text(
        '#include "%s"\n'
        'extern "C" {\n'
        "void row(const uint32_t* w, int i, uint32_t* rows) { pl::rows29_row(w, i, rows); }\n"
        "void mul(int D, int bt, const uint32_t* x, const uint32_t* rows, uint32_t* t) {\n"
        "  if (D == 1 && !bt) pl::rows29<1, false>(x, rows, t);\n"
        "  if (D == 1 && bt) pl::rows29<1, true>(x, rows, t);\n"
        "  if (D == 2 && !bt) pl::rows29<2, false>(x, rows, t);\n"
        "  if (D == 2 && bt) pl::rows29<2, true>(x, rows, t);\n"
        "}\n}\n" % os.path.abspath(os.path.join(CSRC, "fr29.hpp")))
    so = d / "r.so"
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-Wno-unknown-pragmas", str(src), "-o", str(so)])
    lib = ctypes.CDLL(str(so))

    class Lib:
        @staticmethod
        def table(w, D):
            t = (U * 81)()
            for i in range(9):
                v = w * (1 << (29 * (i + D))) % R
                lib.row((U * 8)(*[(v >> (32 * k)) & 0xFFFFFFFF for k in range(8)]), i, t)
            return t

        @staticmethod
        def mul(D, bt, x, t):
            o = (U * 9)()
            lib.mul(D, int(bt), (U * 9)(*[l & 0xFFFFFFFF for l in x]), t, o)
            return [v - (1 << 32) if v >> 31 else v for v in o]

    return Lib


def value(l):
    return sum(d << (29 * i) for i, d in enumerate(l))


def test_table_rows_are_centred_balanced_digits(rows):
    rng = random.Random(1)
    for w in [0, 1, R - 1, R // 2, R // 2 + 1] + [rng.randrange(R) for _ in range(50)]:
        for D in (1, 2):
            t = [v - (1 << 32) if v >> 31 else v for v in rows.table(w, D)]
            assert all(-(1 << 28) <= v <= (1 << 28) for v in t)
            for i in range(9):
                W = value([t[9 * j + i] for j in range(9)])
                assert W % R == w * (1 << (29 * (i + D))) % R and abs(W) < 0.51 * R


@pytest.mark.parametrize("D", [1, 2])
@pytest.mark.parametrize("bt", [False, True])
def test_product_matches_integers(rows, D, bt):
    rng = random.Random(10 * D + bt)
    lo, hi = (-(1 << 28), (1 << 28)) if bt else (0, 1 << 29)
    lim = 1 << 31 if D == 2 else 1 << 30
    ws = [0, 1, R - 1, R // 2] + [rng.randrange(R) for _ in range(40)]
    xs = [[lim - 1] * 9, [-lim] * 9, [lim - 1, -lim] * 4 + [lim - 1], [0] * 9, [1] + [0] * 8, [0] * 8 + [-lim]]
    for w in ws:
        t = rows.table(w, D)
        # every column at its largest: x_i of the sign of W_{i,j}
        worst = []
        for j in range(9):
            s = [v - (1 << 32) if v >> 31 else v for v in t[9 * j:9 * j + 9]]
            worst += [[lim - 1 if v >= 0 else -lim for v in s], [-lim if v >= 0 else lim - 1 for v in s]]
        for x in xs + worst + [[rng.randrange(-lim, lim) for _ in range(9)] for _ in range(40)]:
            o = rows.mul(D, bt, x, t)
            assert value(o) % R == value(x) * w % R, (x, w)
            assert all(lo <= v < hi for v in o[:8]), o
            X = sum(map(abs, x)) / (1 << (29 * D)) * 0.51
            assert -(X + 1.001) * R < value(o) < (X + 0.001) * R


def brev3(k):
    return (k & 1) << 2 | (k & 2) | k >> 2


@pytest.mark.parametrize("inverse", [False, True])
def test_dft8_four_products(rows, inverse):
    """dft_dif<3>'s sequence: exact, every limb within 32 bits, values within
    its stated bound, for random and extreme balanced digits."""
    w = pow(7, (R - 1) >> 3, R)
    if inverse:
        w = pow(w, R - 2, R)
    half = (R + 1) // 2
    i_, c1, c2 = (rows.table(c % R, 1) for c in (w * w, (w + w ** 3) * half, (w - w ** 3) * half))
    rng = random.Random(8 + inverse)
    B = 1 << 28

    def fit(v):
        assert all(-(1 << 31) <= d < (1 << 31) for d in v), v
        return v

    def bfly(x, a, b):
        s, d = fit([p + q for p, q in zip(x[a], x[b])]), fit([p - q for p, q in zip(x[a], x[b])])
        x[a], x[b] = s, d

    def dft(x):
        for i in range(4):
            bfly(x, i, i + 4)
        bfly(x, 0, 2)
        bfly(x, 1, 3)
        bfly(x, 0, 1)
        x[3] = rows.mul(1, False, x[3], i_)
        bfly(x, 2, 3)
        x[6] = rows.mul(1, False, x[6], i_)
        bfly(x, 4, 6)
        bfly(x, 5, 7)
        x[5] = rows.mul(1, False, x[5], c1)
        x[7] = rows.mul(1, False, x[7], c2)
        bfly(x, 5, 7)
        bfly(x, 4, 5)
        bfly(x, 6, 7)

    tops = [B // 8, -(B // 8)]  # a 256-bit value's top digit is below 2^25
    cases = [[[rng.randrange(-B, B) for _ in range(8)] + [rng.randrange(-(1 << 25), 1 << 25)] for _ in range(8)]
             for _ in range(300)]
    cases += [[[rng.choice([-B, B - 1]) for _ in range(8)] + [rng.choice(tops)] for _ in range(8)] for _ in range(300)]
    cases += [[[s * (B - 1) if s > 0 else -B for _ in range(8)] + [s * (B // 8)] for s in signs]
              for signs in ([1] * 8, [-1] * 8, [1, 1, 1, 1, -1, -1, -1, -1], [1, -1] * 4, [1, 1, -1, -1] * 2)]
    for x in cases:
        v = [value(l) for l in x]
        V = max(map(abs, v))
        dft(x)
        for k in range(8):
            got = value(x[brev3(k)])
            assert got % R == sum(v[j] * pow(w, j * k, R) for j in range(8)) % R, k
            assert abs(got) <= max(8 * V, 2 * V + 26 * R)


def test_generated_columns_current():
    out = subprocess.check_output(["python3", os.path.join(CSRC, "gen_rows29_columns.py")]).decode()
    assert out == open(os.path.join(CSRC, "rows29_columns.inc")).read()
