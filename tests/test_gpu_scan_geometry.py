"""Grand product, batch inversion, evaluation and division at the edges of their block geometries
(256 threads x 1, 2, 4, 8, 16 elements; one and several blocks), against the
oracle, with zeros, ones and r - 1 among the inputs."""
import numpy as np
import pytest

import pyoracle as po

pytestmark = pytest.mark.gpu

MINUS_ONE_INT = [0xFFFFFFFF00000000, 0x53BDA402FFFE5BFE, 0x3339D80809A1D805, 0x73EDA753299D7D48]  # the word r - 1


@pytest.fixture(scope="module")
def pl():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import plffi
    plffi.lib()
    return plffi


def inputs(n, seed):
    x = po.uniform(n, seed)
    x[::7] = MINUS_ONE_INT
    x[3::11] = po.one()[0]
    return x


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 2047, 2048, 2049,
                               4096, 4111, 8193, 4096 * 256, 4096 * 257 + 1])
def test_grand_product_edges(pl, n):
    import torch
    print("gp edge", n, flush=True)
    x = inputs(n, po.seed(po.OP_GP, 1, n & 0xff))
    exp = po.grand_product(x)
    a = pl.to_dev(x)
    incl = torch.zeros_like(a)
    pl.grand_product(a, incl_out=incl)
    np.testing.assert_array_equal(pl.to_host(a), exp)
    gi = pl.to_host(incl)
    np.testing.assert_array_equal(gi[:-1], exp[1:])
    np.testing.assert_array_equal(gi[-1:], po.mul(exp[-1:], x[-1:]))


@pytest.mark.parametrize("n", [1, 2, 63, 65, 255, 256, 257, 512, 513, 1024, 1025, 2047, 2048, 2049, 4097,
                               2048 * 256 + 1, 2048 * 1025])
def test_inverse_and_quotient_edges(pl, n):
    print("inv edge", n, flush=True)
    x, y = inputs(n, n), po.uniform(n, n + 1)
    x[n // 2] = 0
    x[-1 if n > 1 else 0] = 0
    inv = np.zeros_like(x)
    po.lib().or_vec_inv(po.P(inv), po.P(x), n)
    xd, yd = pl.to_dev(x), pl.to_dev(y)
    np.testing.assert_array_equal(pl.to_host(pl.vec_op("inv", xd)), inv)
    np.testing.assert_array_equal(pl.to_host(pl.vec_op("div", yd, xd)), po.mul(y, inv))
    # in place over the divisor and over the numerator
    a, b = pl.to_dev(x), pl.to_dev(y)
    np.testing.assert_array_equal(pl.to_host(pl.vec_op("div", b, a, out=a)), po.mul(y, inv))
    np.testing.assert_array_equal(pl.to_host(pl.vec_op("div", b, xd, out=b)), po.mul(y, inv))


# single blocks of each geometry, the latency form's smallest sizes, its largest
# and the first above it (last wave's runs cut inside and at a chunk of four
# elements), a second level of one and of several blocks
@pytest.mark.parametrize("n", [1, 255, 256, 257, 512, 513, 1024, 1025, 2048, 2049, 2052, 3071, 4095, 4097,
                               255 * 256 * 28, 255 * 256 * 28 + 1, 2000003, 2000004, 2000015, 2000017,
                               4096 * 512 + 1, 4096 * 1025, 4096 * 2049 - 3, 4096 * 4096 + 1])
def test_evaluation_and_division_edges(pl, n):
    import torch
    print("eval/div edge", n, flush=True)
    x, z = inputs(n, n), po.uniform(1, n + 7)
    q, r = po.div(x, z)
    xd, zd = pl.to_dev(x), pl.to_dev(z)
    np.testing.assert_array_equal(pl.to_host(pl.evaluate(xd, zd)), po.eval_(x, z))
    rem = torch.zeros((1, 4), dtype=torch.int64, device="cuda")
    pl.div_linear(xd, zd, rem=rem)
    np.testing.assert_array_equal(pl.to_host(xd), q)
    np.testing.assert_array_equal(pl.to_host(rem).reshape(-1), np.asarray(r).reshape(-1))


# a top level with its own launch (more than 256 block products), and around the
# row counts where one block of run products hands over to two levels
@pytest.mark.parametrize("lg", [13, 14, 23])
def test_perm_grand_product_is_the_ratios_product(pl, lg):
    print("perm gp levels", lg, flush=True)
    n = 1 << lg
    k = np.concatenate([po.from_u64(v) for v in (1, 7, 13)])
    col = [pl.to_dev(po.uniform(n, po.seed(po.OP_GP, lg, 60 + j))) for j in range(6)]
    beta, gamma = pl.to_dev(po.uniform(1, 5)), pl.to_dev(po.uniform(1, 6))
    col[3][n // 3] = 0
    dom = pl.Domain(lg)
    ratio = pl.perm_ratio(col[:3], col[3:], beta, gamma, k, dom)
    z = pl.perm_ratio(col[:3], col[3:], beta, gamma, k, dom, grand_product=True)
    np.testing.assert_array_equal(pl.to_host(z), pl.to_host(pl.grand_product(ratio)))
