"""Plain digits in the NTT passes (csrc/fr29.hpp mont29_word, csrc/ntt_pass.hpp
dft_dif): the twiddle product that leaves a 256-bit word and the eight-point
DFT of digits in [0, 2^29), on the host against Python integers at the limits;
the passes on the GPU against the oracle for words up to 2^256 - 1."""
import ctypes
import os
import random
import subprocess

import numpy as np
import pytest

import pyoracle as po

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "ppopp26-artifact_amd", "csrc")
R = 0x73EDA753299D7D483339D80809A1D80553BDA402FFFE5BFEFFFFFFFF00000001
M = 1 << 29
U = ctypes.c_uint32


def value(l):
    return sum(d << (29 * i) for i, d in enumerate(l))


def signed(v):
    return v - (1 << 32) if v >> 31 else v


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("plain")
    src = d / "p.cpp"
    src.write_text(
        '#include "%s"\n'
        'extern "C" {\n'
        "void word(const uint32_t* a, const uint32_t* w, uint32_t* t) { pl::mont29_word(a, w, t); }\n"
        "void pbd(const uint32_t* w, uint32_t* x) { pl::to_pbd(w, x); }\n"
        "void unpack(const uint32_t* x, uint32_t* b) { pl::pbd_unpack(x, b); }\n"
        "void row(const uint32_t* w, int i, uint32_t* rows) { pl::rows29_row(w, i, rows); }\n"
        "void rows1(const uint32_t* x, const uint32_t* rows, uint32_t* t) { pl::rows29<1, false>(x, rows, t); }\n"
        "}\n" % os.path.abspath(os.path.join(CSRC, "fr29.hpp")))
    so = d / "p.so"
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-Wno-unknown-pragmas", str(src), "-o", str(so)])
    return ctypes.CDLL(str(so))


def factor(lib, w):
    x, b = (U * 8)(), (U * 9)()
    lib.pbd((U * 8)(*[(w >> (32 * k)) & 0xFFFFFFFF for k in range(8)]), x)
    lib.unpack(x, b)
    return b


@pytest.mark.parametrize("top", [30, 17, 1, 0, -1, -17, -30])
def test_twiddle_product_leaves_a_word(lib, top):
    # limbs anywhere in 32 bits, value within about top r (30.4 r is the DFT's largest)
    rng = random.Random(100 + top)
    lim = (1 << 31) - 1
    inv = pow(1 << 261, R - 2, R)
    for w in [0, 1, R - 1, R // 2, R // 2 + 1] + [rng.randrange(R) for _ in range(60)]:
        b = factor(lib, w)
        bs = [signed(v) for v in b]
        rows = [[lim] * 8, [-lim] * 8, [0] * 8, [lim if v >= 0 else -lim for v in bs[:8]],
                [-lim if v >= 0 else lim for v in bs[7::-1]]]
        for lo in rows + [[rng.randrange(-lim, lim + 1) for _ in range(8)] for _ in range(8)]:
            x = lo + [top * R >> 232]
            t = (U * 9)()
            lib.word((U * 9)(*[v & 0xFFFFFFFF for v in x]), b, t)
            t = list(t)
            assert all(v < M for v in t[:8]) and t[8] < 1 << 24, t  # joins to 256 bits
            assert value(t) % R == value(x) * value(bs) * inv % R
            assert value(t) > 0


@pytest.mark.parametrize("inverse", [False, True])
def test_dft8_plain_digits(lib, inverse):
    w = pow(7, (R - 1) >> 3, R)
    if inverse:
        w = pow(w, R - 2, R)
    half = (R + 1) // 2

    def table(c):
        t = (U * 81)()
        for i in range(9):
            v = c * (1 << (29 * (i + 1))) % R
            lib.row((U * 8)(*[(v >> (32 * k)) & 0xFFFFFFFF for k in range(8)]), i, t)
        return t

    i_, c1, c2 = (table(c % R) for c in (w * w, (w + w ** 3) * half, (w - w ** 3) * half))

    def mul(x, t):
        assert all(abs(v) <= 1 << 30 for v in x)
        o = (U * 9)()
        lib.rows1((U * 9)(*[v & 0xFFFFFFFF for v in x]), t, o)
        return [signed(v) for v in o]

    def fit(v):
        assert all(-(1 << 31) <= d < (1 << 31) for d in v), v
        return v

    def bfly(x, a, b):
        x[a], x[b] = [p + q for p, q in zip(x[a], x[b])], fit([p - q for p, q in zip(x[a], x[b])])

    def dft(x):
        for i in range(4):
            bfly(x, i, i + 4)
        bfly(x, 0, 2)
        bfly(x, 1, 3)
        bfly(x, 0, 1)
        x[0] = fit([x[0][0] - (1 << 31)] + [v + 4 - (1 << 31) for v in x[0][1:8]] + [x[0][8] + 4])
        x[3] = mul(x[3], i_)
        bfly(x, 2, 3)
        x[6] = mul(x[6], i_)
        bfly(x, 4, 6)
        bfly(x, 5, 7)
        x[5], x[7] = mul(x[5], c1), mul(x[7], c2)
        bfly(x, 5, 7)
        bfly(x, 4, 5)
        bfly(x, 6, 7)
        for v in x:
            fit(v)

    rng = random.Random(9 + inverse)
    lo, hi = [0] * 9, [M - 1] * 8 + [(1 << 24) - 1]
    cases = [[hi] * 8, [lo] * 8] + [[hi if m >> k & 1 else lo for k in range(8)] for m in range(1, 255, 3)]
    cases += [[[rng.randrange(M) for _ in range(8)] + [rng.randrange(-(1 << 24), 1 << 24)] for _ in range(8)]
              for _ in range(40)]
    for c in cases:
        x = [list(v) for v in c]
        dft(x)
        for k in range(8):
            brev = (k & 1) << 2 | (k & 2) | k >> 2
            assert value(x[brev]) % R == sum(value(v) * pow(w, j * k, R) for j, v in enumerate(c)) % R
            assert abs(value(x[brev])) < 30.5 * R


@pytest.mark.gpu
@pytest.mark.parametrize("lg,npoly", [(3, 1 << 16), (4, 1 << 15), (5, 20000), (6, 8200), (8, 2049), (11, 257), (13, 65),
                                      (19, 1)])
def test_passes_any_256_bit_words(lg, npoly):
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import plffi as pl
    n = 1 << lg
    rng = np.random.default_rng(lg)
    ones = rng.integers(0, 2, size=npoly * n, dtype=np.uint64)
    ones[:n] = 1  # the first polynomial: the largest word throughout
    x = np.repeat((0 - ones)[:, None], 4, axis=1)
    v = ((1 << 256) - 1) % R
    word = np.array([(v >> (64 * i)) & 0xFFFFFFFFFFFFFFFF for i in range(4)], dtype=np.uint64)
    y = np.where(ones[:, None] != 0, word[None, :], np.uint64(0))
    dom = pl.Domain(lg)
    print("pass words lg", lg, "npoly", npoly, flush=True)
    for inverse in (False, True):
        out = pl.to_host(pl.ntt_batch(pl.to_dev(x), dom, npoly, inverse=inverse))
        for p in {0, 1 % npoly, npoly // 2, npoly - 1}:
            np.testing.assert_array_equal(out[p * n:(p + 1) * n], po.ntt(y[p * n:(p + 1) * n], lg, inverse=inverse))
