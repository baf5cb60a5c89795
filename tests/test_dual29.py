"""The two products under one reduction of the small transforms' radix-4 step
(dual29 in csrc/fr29.hpp, csrc/ntt_lane.hip) on the host against Python
integers: congruence, ranges and column sums at the limits."""
import ctypes
import os
import random
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "ppopp26-artifact_amd", "csrc")
R = 0x73EDA753299D7D483339D80809A1D80553BDA402FFFE5BFEFFFFFFFF00000001
RD = [(R >> (29 * i)) & ((1 << 29) - 1) for i in range(9)]
M = 1 << 29
U = ctypes.c_uint32


def value(l):
    return sum(d << (29 * i) for i, d in enumerate(l))


def signed(v):
    return v - (1 << 32) if v >> 31 else v


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("dual29")
    src = d / "d.cpp"
    src.write_text(
        '#include "%s"\n'
        'extern "C" {\n'
        "void dual(int word, const uint32_t* a, const uint32_t* w, const uint32_t* b, const uint32_t* v, uint32_t* t) {\n"
        "  if (word) pl::dual29<true>(a, w, b, v, t); else pl::dual29<false>(a, w, b, v, t);\n"
        "}\n"
        "void pbd(const uint32_t* w, uint32_t* x) { pl::to_pbd(w, x); }\n"
        "void unpack(const uint32_t* x, uint32_t* b) { pl::pbd_unpack(x, b); }\n"
        "void split(const uint32_t* x, uint32_t* a) { pl::split29(x, a); }\n"
        "}\n" % os.path.abspath(os.path.join(CSRC, "fr29.hpp")))
    so = d / "d.so"
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-Wno-unknown-pragmas", str(src), "-o", str(so)])
    return ctypes.CDLL(str(so))


def word8(w):
    return (U * 8)(*[(w >> (32 * k)) & 0xFFFFFFFF for k in range(8)])


def factor(lib, w):
    """balanced digits of a table factor w < r"""
    x, b = (U * 8)(), (U * 9)()
    lib.pbd(word8(w), x)
    lib.unpack(x, b)
    return [signed(v) for v in b]


def split(lib, x):
    a = (U * 9)()
    lib.split(word8(x), a)
    return list(a)


def dual(lib, word, a, w, b, v):
    # the columns beside it, without a width
    m, acc = [], 0
    for k in range(17):
        for i in range(max(0, k - 8), min(k, 8) + 1):
            acc += a[i] * w[k - i] + b[i] * v[k - i]
            assert -(1 << 63) <= acc < 1 << 63
        for i in range(max(0, k - 8), min(k, 8) + 1):
            if i < k:
                acc -= m[i] * RD[k - i]
                assert -(1 << 63) <= acc < 1 << 63
        d = acc % M
        if word and k == 8:
            d = (d - M if d >= M // 2 else d) - M
        if k <= 8:
            m.append(d)
        acc = (acc - d) >> 29
    t = (U * 9)()
    arr = lambda l: (U * 9)(*[x & 0xFFFFFFFF for x in l])  # noqa: E731
    lib.dual(int(word), arr(a), arr(w), arr(b), arr(v), t)
    return [signed(x) for x in t]


@pytest.mark.parametrize("word", [False, True])
def test_limits(lib, word):
    rng = random.Random(31 + word)
    lim = (1 << 30) - 1
    inv = pow(1 << 261, -1, R)
    ws = [0, 1, R - 1, R // 2] + [rng.randrange(R) for _ in range(20)]
    for w, v in [(w, v) for w in ws for v in ws[::5] + [rng.randrange(R)]]:
        W, V = factor(lib, w), factor(lib, v)
        # every product of a column of one sign: limbs by the digits they meet in the largest column
        aw, bv = [lim if d >= 0 else -lim for d in W[::-1]], [lim if d >= 0 else -lim for d in V[::-1]]
        pairs = [(aw, bv), ([-x for x in aw], [-x for x in bv]), ([lim] * 9, [-lim] * 9), ([lim] * 9, [lim] * 9)]
        pairs += [([rng.randrange(-lim, lim + 1) for _ in range(9)], [rng.choice((-lim, lim)) for _ in range(9)])]
        for a, b in pairs:
            t = dual(lib, word, a, W, b, V)
            T = value(a) * value(W) + value(b) * value(V)
            assert (value(t) - T * inv) % R == 0
            assert all(0 <= d < M for d in t[:8])
            lo, hi = (T * 2 + (R << 261), T * 2 + (3 * R << 261)) if word else (T - (R << 261), T)
            s = value(t) << (262 if word else 261)
            assert lo - (1 << 262) < s <= hi + (1 << 262)


@pytest.mark.parametrize("inverse", [False, True])
def test_radix4_steps(lib, inverse):
    """Two radix-4 steps and the twiddle product between launches, as the lanes
    of a quad form them: limbs, ranges and values."""
    i4 = pow(7, (R - 1) >> 2, R)
    if inverse:
        i4 = pow(i4, R - 2, R)
    R261 = (1 << 261) % R
    rng = random.Random(41 + inverse)
    top = (1 << 256) - 1

    def step(x, tw, word):
        out = []
        for k in range(4):
            # lanes 0, 1 hold x_q + x_(q+2), lanes 2, 3 x_(q-2) - x_q; lane k takes the pairs of its parity
            u = [p + q if k % 2 == 0 else p - q for p, q in zip(x[0], x[2])]
            v = [p + q if k % 2 == 0 else p - q for p, q in zip(x[1], x[3])]
            assert all(abs(d) < 1 << 30 for d in u + v)
            out.append(dual(lib, word, u, factor(lib, tw[k] * R261 % R), v,
                            factor(lib, tw[k] * pow(i4, k, R) * R261 % R)))
        return out

    def expect(x, tw):
        return [tw[k] * sum(x[j] * pow(i4, j * k, R) for j in range(4)) % R for k in range(4)]

    cases = [[top if m >> j & 1 else 0 for j in range(4)] for m in range(16)]
    cases += [[rng.randrange(1 << 256) for _ in range(4)] for _ in range(60)]
    for c in cases:
        tw = [[rng.choice((1, R - 1, rng.randrange(R))) for _ in range(4)] for _ in range(3)]
        y = step([split(lib, v) for v in c], tw[0], False)
        want = expect(c, tw[0])
        for t, e in zip(y, want):
            assert value(t) % R == e and -1126 * R < 1000 * value(t) < 126 * R
        y = step(y, tw[1], False)  # a later step: digits plain, the top signed
        want = expect(want, tw[1])
        for t, e in zip(y, want):
            assert value(t) % R == e and -1070 * R < 1000 * value(t) < 70 * R
        y = step(y, tw[2], True)  # stored between the launches
        want = expect(want, tw[2])
        for t, e in zip(y, want):
            assert value(t) % R == e and 430 * R < 1000 * value(t) < 1570 * R
            assert all(0 <= d < M for d in t[:8]) and 0 <= t[8] < 1 << 24
