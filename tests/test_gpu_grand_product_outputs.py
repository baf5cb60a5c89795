"""Both outputs of the grand product given the same buffer: the exclusive
products are what stays."""
import numpy as np
import pytest

import pyoracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 300, 4096, 5000, 4096 * 257 + 1])
@pytest.mark.parametrize("noalloc", [False, True])
def test_one_buffer(n, noalloc):
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import plffi as pl
    x = po.uniform(n, po.seed(po.OP_GP, 2, n & 0xff))
    print("grand product, outputs in one buffer", n, noalloc, flush=True)
    a = pl.to_dev(x)
    (pl.grand_product_noalloc if noalloc else pl.grand_product)(a, incl_out=a)
    np.testing.assert_array_equal(pl.to_host(a), po.grand_product(x))
