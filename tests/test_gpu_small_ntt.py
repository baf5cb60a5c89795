"""The one-element-per-lane form of small transforms (csrc/ntt_lane.hip)
against the oracle: every size, odd batch sizes, both directions, in place,
with coset factors and interleaved outputs, and extreme input words."""
import numpy as np
import pytest

import pyoracle as po

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pl():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import plffi
    plffi.lib()
    return plffi


@pytest.mark.parametrize("lg", range(4, 20))
def test_every_size(pl, lg):
    n = 1 << lg
    dom = pl.Domain(lg)
    for npoly in (1, 3) if lg > 8 else (1, 3, 7, 17, 65):
        x = po.uniform(npoly * n, po.seed(po.OP_NTT, lg, npoly))
        x[0] = 0
        x[-1] = [0xFFFFFFFF00000000, 0x53BDA402FFFE5BFE, 0x3339D80809A1D805, 0x73EDA753299D7D48]  # r - 1
        for inverse in (False, True):
            print("lane form lg", lg, "npoly", npoly, "inverse", inverse, flush=True)
            ref = np.concatenate([po.ntt(x[p * n:(p + 1) * n], lg, inverse=inverse) for p in range(npoly)])
            xd = pl.to_dev(x)
            np.testing.assert_array_equal(pl.to_host(pl.ntt_batch(xd, dom, npoly, inverse=inverse)), ref)
            np.testing.assert_array_equal(pl.to_host(xd), x)
            pl.ntt_batch(xd, dom, npoly, inverse=inverse, out=xd)  # in place
            np.testing.assert_array_equal(pl.to_host(xd), ref)


@pytest.mark.parametrize("lg,lb", [(4, 1), (7, 2), (9, 3), (10, 2), (11, 1), (12, 2), (13, 4), (15, 2)])
def test_lde(pl, lg, lb):
    c = po.uniform(1 << lg, po.seed(po.OP_LDE, lg, lb))
    ref = po.lde(c, lg, lb, po.ref_lde_shift(lb))
    dom = pl.LdeDomain(lg, lb)
    print("lane form lde", lg, lb, flush=True)
    np.testing.assert_array_equal(pl.to_host(pl.lde(pl.to_dev(c), dom)), ref)
    import torch
    buf = torch.zeros((1 << (lg + lb), 4), dtype=torch.int64, device="cuda")  # output over its own input
    buf[:1 << lg] = pl.to_dev(c)
    np.testing.assert_array_equal(pl.to_host(pl.lde(buf[:1 << lg], dom, out=buf)), ref)


def test_any_256_bit_words(pl):
    # inputs need not be canonical: words up to 2^256 - 1 reduce to their class
    for lg in (5, 10, 12, 15):
        n = 1 << lg
        x = np.full((n, 4), 0xFFFFFFFFFFFFFFFF, dtype=np.uint64)
        x[::3] = 0
        R = 0x73EDA753299D7D483339D80809A1D80553BDA402FFFE5BFEFFFFFFFF00000001
        v = ((1 << 256) - 1) % R
        y = x.copy()
        y[x[:, 0] != 0] = [(v >> (64 * i)) & 0xFFFFFFFFFFFFFFFF for i in range(4)]
        dom = pl.Domain(lg)
        for inverse in (False, True):
            np.testing.assert_array_equal(pl.to_host(pl.ntt(pl.to_dev(x), dom, inverse=inverse)),
                                          po.ntt(y, lg, inverse=inverse))


@pytest.mark.parametrize("lg", [4, 5, 8, 9, 10, 11, 14, 17, 18])
def test_coset_inverse(pl, lg):
    # the coset powers ride on the last step's factors
    for shift in (None, po.uniform(1, 99)):
        dom = pl.CosetDomain(lg, shift)
        g = po.from_u64(7) if shift is None else shift
        x = po.uniform(1 << lg, po.seed(po.OP_INTT, lg, 3))
        print("lane form inverse coset", lg, flush=True)
        xd = pl.to_dev(x)
        ref = po.coset_intt(x, lg, g)
        np.testing.assert_array_equal(pl.to_host(pl.coset_ntt(xd, dom, inverse=True)), ref)
        pl.coset_ntt(xd, dom, inverse=True, out=xd)
        np.testing.assert_array_equal(pl.to_host(xd), ref)
