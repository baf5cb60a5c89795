"""The arithmetic of an NTT pass (csrc/ntt_pass.hpp) and of the permutation
terms (csrc/ops.hip) as the kernels do it now, on the host
(tests/native/pass_column.cpp) against Python integers: plain digits, the
four-product DFT_8 with its zero in mixed digits, inner twiddles and beta as
rows, the reductions of the elements without a twiddle, the twiddle product that
leaves a word, and passes chained into a whole transform.  Every limb, column
and word bound is checked at the limits of the input words."""
import ctypes
import os
import random
import re
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "ppopp26-artifact_amd", "csrc")
R = 0x73EDA753299D7D483339D80809A1D80553BDA402FFFE5BFEFFFFFFFF00000001
TOP = (1 << 256) - 1
M = 1 << 29
R256, R261 = (1 << 256) % R, (1 << 261) % R
U = ctypes.c_uint32


def words(vals):
    return (U * (8 * len(vals)))(*[(v >> (32 * i)) & 0xFFFFFFFF for v in vals for i in range(8)])


def ints(a):
    return [sum(a[8 * k + i] << (32 * i) for i in range(8)) for k in range(len(a) // 8)]


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = tmp_path_factory.mktemp("pass_column") / "p.so"
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-Wno-unknown-pragmas", "-I",
                           os.path.abspath(CSRC), os.path.join(HERE, "native", "pass_column.cpp"), "-o", str(so)])
    return ctypes.CDLL(str(so))


def pbd(lib, vals):
    """pbd words of table factors v R'"""
    out = (U * (8 * len(vals)))()
    for k, v in enumerate(vals):
        x = (U * 8)()
        lib.t_to_pbd(words([v * R261 % R]), x)
        out[8 * k:8 * k + 8] = list(x)
    return out


def rows(lib, ws, D):
    out = []
    for w in ws:
        t = (U * 81)()
        for i in range(9):
            lib.t_row(words([w * pow(2, 29 * (i + D), R) % R]), i, t)
        out += list(t)
    return (U * len(out))(*out)


def root(lg, inverse):
    w = pow(7, (R - 1) >> lg, R)
    return pow(w, R - 2, R) if inverse else w


class Column:
    """the pass's tables for one direction, and one column through the model"""

    def __init__(self, lib, inverse):
        self.lib, self.inverse = lib, inverse
        w8, w64, half = root(3, inverse), root(6, inverse), (R + 1) // 2
        self.f = rows(lib, [w8 * w8 % R, (w8 + w8 ** 3) * half % R, (w8 - w8 ** 3) * half % R], 1)
        self.inner = rows(lib, [pow(w64, e, R) for e in range(64)], 2)

    def run(self, x, premul=None, tw=None, scale=None):
        la = len(x).bit_length() - 4
        out = (U * (8 * len(x)))()
        opt = lambda v: pbd(self.lib, v) if v is not None else None  # noqa: E731
        bad = self.lib.t_column(la, words(x), self.f, self.inner, opt(premul), opt(tw),
                                opt([scale]) if scale is not None else None, out)
        assert bad == 0, (la, self.inverse)
        y = ints(out)
        if tw is not None:
            assert all(6 * R < 100 * v < 194 * R for v in y)
        else:
            assert all(v < R for v in y)
        return y

    def dft(self, x):
        w = root(len(x).bit_length() - 1, self.inverse)
        return [sum(v * pow(w, j * k, R) for j, v in enumerate(x)) % R for k in range(len(x))]


ALTERNATING = sum((M - 1) << (58 * i) for i in range(5)) & TOP  # every other digit full


def inputs(rng, n):
    yield [TOP] * n
    yield [0] * n
    yield [ALTERNATING if j & 1 else TOP ^ ALTERNATING for j in range(n)]
    # full and empty words by the bits of their index: sums and differences of
    # every butterfly level at their limits, of one sign
    for bits in range(1, n):
        if n <= 16 or bits in (1, 2, 4, 8, 16, 32, 3, 5, 6, 7, 9, 24, 40, 56, 63):
            yield [TOP if bin(j & bits).count("1") & 1 else 0 for j in range(n)]
    for _ in range(6):
        yield [rng.choice((0, R - 1, R, 2 * R, TOP)) for _ in range(n)]
    for _ in range(6):
        yield [rng.randrange(1 << 256) for _ in range(n)]


@pytest.mark.parametrize("la", [0, 1, 2, 3])
@pytest.mark.parametrize("inverse", [False, True])
def test_column(lib, la, inverse):
    rng = random.Random(10 * la + inverse)
    n = 8 << la
    col = Column(lib, inverse)
    for i, x in enumerate(inputs(rng, n)):
        X = col.dft(x)
        tw = [rng.choice((0, 1, R - 1, rng.randrange(R))) for _ in range(n)]
        y = col.run(x, tw=tw)
        assert all((v - e * t) % R == 0 for v, e, t in zip(y, X, tw))
        assert col.run(x) == X
        s = rng.randrange(R)
        if i % 2:
            assert col.run(x, scale=s) == [e * s % R for e in X]
        else:
            pm = [rng.randrange(R) for _ in range(n)]
            P = col.dft([v * p % R for v, p in zip(x, pm)])
            y = col.run(x, premul=pm, tw=tw)
            assert all((v - e * t) % R == 0 for v, e, t in zip(y, P, tw))


def transform(lib, x, split, inverse):
    """a whole transform as the passes run it: pass p on the columns of each
    sub-problem with its twiddles, the words handed on as they are"""
    col = Column(lib, inverse)
    lg = sum(split)
    n_inv = pow(1 << lg, R - 2, R) if inverse else 1

    def solve(v, ms, scale):
        if len(ms) == 1:
            return col.run(v, scale=scale if len(split) == 1 and inverse else None)
        size = len(v)
        M1, S = 1 << ms[0], size >> ms[0]
        w = root(size.bit_length() - 1, inverse)
        cols = [col.run([v[j + S * r] for r in range(M1)], tw=[pow(w, j * k, R) * scale % R for k in range(M1)])
                for j in range(S)]
        out = [0] * size
        for k in range(M1):
            for i, e in enumerate(solve([cols[j][k] for j in range(S)], ms[1:], 1)):
                out[k + M1 * i] = e
        return out

    return solve(x, split, n_inv)


@pytest.mark.parametrize("split", [(6,), (3, 3), (4, 5), (6, 3), (3, 3, 3)])
@pytest.mark.parametrize("inverse", [False, True])
def test_chained_passes(lib, split, inverse):
    rng = random.Random(sum(split) + inverse)
    lg = sum(split)
    n = 1 << lg
    w = root(lg, inverse)
    f = pow(n, R - 2, R) if inverse else 1
    for x in ([TOP] * n, [TOP if j & 1 else 0 for j in range(n)], [rng.randrange(1 << 256) for _ in range(n)]):
        pw = [pow(w, e, R) for e in range(n)]
        ks = rng.sample(range(n), 40) + [0, 1, n // 2, n - 1]
        y = transform(lib, x, split, inverse)
        for k in ks:
            assert y[k] == f * sum(v * pw[j * k % n] for j, v in enumerate(x)) % R


def row_shift():
    text = open(os.path.join(CSRC, "fr29.hpp")).read()
    body = text[text.index("kRowShift[2][9][9] = {"):]
    v = [int(h, 16) for h in re.findall(r"0x([0-9a-f]+)u", body[:body.index(";")])]
    assert len(v) == 162
    return v


def test_row_shift_factors():
    s = [v - (1 << 32) if v >> 31 else v for v in row_shift()]
    for rp in (0, 1):
        for i in range(9):
            d = s[81 * rp + 9 * i:81 * rp + 9 * i + 9]
            assert all(-(1 << 28) <= v <= 1 << 28 for v in d)
            assert sum(v << (29 * j) for j, v in enumerate(d)) % R == pow(2, 29 * (i + 2) + (0 if rp else 5), R)


def test_perm_terms(lib):
    shift = (U * 81)(*row_shift()[:81])
    rng = random.Random(21)
    inv = pow(R256, -1, R)
    f = lambda x: x * inv % R  # noqa: E731
    for trial in range(400):
        pick = (lambda: TOP) if trial < 4 else (lambda: rng.choice((0, R - 1, TOP))) if trial < 120 else \
               (lambda: rng.randrange(1 << 256))
        w0, w1, beta = (rng.choice((0, 1, R - 1, rng.randrange(R))) for _ in range(3))  # canonical: tables and a challenge
        gamma, *v = (pick() for _ in range(7))
        ws, ss = v[:3], v[3:]
        sk = trial % 2
        k = [1, 7, 13] if sk else [rng.randrange(R) for _ in range(3)]
        num_out, den_out = (U * 8)(), (U * 8)()
        bad = lib.t_perm_terms(words([w0]), words([w1]), words([beta]), words([32 * beta % R]), words([gamma]), shift,
                               pbd(lib, [32 * kj % R for kj in k]), sk, words(ws), words(ss), num_out, den_out)
        assert bad == 0, trial
        wi, num, den = f(w0) * f(w1), pow(1024, -1, R), pow(1024, -1, R)
        for j in range(3):
            num = num * (f(ws[j]) + f(gamma) + f(beta) * k[j] * wi) % R
            den = den * (f(ws[j]) + f(gamma) + f(beta) * f(ss[j])) % R
        assert ints(num_out) == [num * R256 % R] and ints(den_out) == [den * R256 % R]
