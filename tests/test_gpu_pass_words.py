"""The words between pl_ntt_pass calls: ordinary 256-bit integers congruent to
the elements and below 1.94 r, so that a caller may reduce them, or add r, and
the next pass gives the same."""
import numpy as np
import pytest

import pyoracle as po

pytestmark = pytest.mark.gpu

R = 0x73EDA753299D7D483339D80809A1D80553BDA402FFFE5BFEFFFFFFFF00000001
M64 = (1 << 64) - 1


def ints(a):
    return [int(w[0]) | int(w[1]) << 64 | int(w[2]) << 128 | int(w[3]) << 192 for w in a]


def words(v):
    return np.array([[(x >> (64 * i)) & M64 for i in range(4)] for x in v], dtype=np.uint64)


@pytest.mark.parametrize("lg", [7, 10, 13])
@pytest.mark.parametrize("inverse", [False, True])
def test_words_between_passes(lg, inverse):
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import plffi as pl
    dom = pl.Domain(lg)
    x = po.uniform(1 << lg, po.seed(po.OP_NTT, lg, 5))
    x[1] = M64  # the largest word
    y = x.copy()
    y[1] = words([((1 << 256) - 1) % R])[0]
    ref = po.ntt(y, lg, inverse=inverse)
    passes = pl.lib().pl_domain_num_passes(dom.h)
    assert passes > 1
    for change in (lambda v: v, lambda v: v % R, lambda v: v % R + R):
        print("words between passes", lg, inverse, flush=True)
        d = pl.to_dev(x)
        for p in range(passes - 1):
            mid = ints(pl.to_host(pl.ntt_pass(d, torch.empty_like(d), dom, p, inverse=inverse)))
            assert all(v * 100 < 194 * R for v in mid)
            d = pl.to_dev(words([change(v) for v in mid]))
        out = pl.ntt_pass(d, torch.empty_like(d), dom, passes - 1, inverse=inverse)
        np.testing.assert_array_equal(pl.to_host(out), ref)
