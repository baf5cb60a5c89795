"""Grand product of words that are not canonical: any 256-bit word stands for
its class, wherever it falls in a thread's run."""
import numpy as np
import pytest

import pyoracle as po

pytestmark = pytest.mark.gpu

R = 0x73EDA753299D7D483339D80809A1D80553BDA402FFFE5BFEFFFFFFFF00000001
M64 = (1 << 64) - 1


def words(v):
    return np.array([[(x >> (64 * i)) & M64 for i in range(4)] for x in v], dtype=np.uint64)


# one value per thread, two, four, eight and sixteen; several blocks; a second level
@pytest.mark.parametrize("n", [5, 256, 511, 1000, 2048, 4093, 4096 * 3 + 7, 4096 * 257 + 1])
@pytest.mark.parametrize("kind", ["largest", "one in seven", "first of a run", "last of a run", "multiples of r"])
def test_any_256_bit_words(n, kind):
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import plffi as pl
    x = po.uniform(n, po.seed(po.OP_GP, 1, n & 0xff))
    at = {"largest": slice(None), "one in seven": slice(3, None, 7), "first of a run": slice(0, None, 16),
          "last of a run": slice(15 if n > 15 else 0, None, 16), "multiples of r": slice(n - n // 8 - 1, None, 5)}[kind]
    y, z = x.copy(), x.copy()
    idx = np.arange(n)[at]
    if kind == "multiples of r":
        v = [R * (1 + int(i) % 2) for i in idx]
    else:
        # from the top of the range down to just above r, by steps that no block size divides
        v = [(1 << 256) - 1 - (int(i) % 1009) * (((1 << 256) - 1 - R) // 1009) for i in idx]
    z[at] = words(v)
    y[at] = words([a % R for a in v])
    print("grand product words", n, kind, flush=True)
    exp = po.grand_product(y)
    a = pl.to_dev(z)
    incl = torch.zeros_like(a)
    pl.grand_product(a, incl_out=incl)
    np.testing.assert_array_equal(pl.to_host(a), exp)
    gi = pl.to_host(incl)
    np.testing.assert_array_equal(gi[:-1], exp[1:])
    np.testing.assert_array_equal(gi[-1:], po.mul(exp[-1:], y[-1:]))
