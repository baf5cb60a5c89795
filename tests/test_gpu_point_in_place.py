"""Opening and division whose results lie over the point: the point is read
before anything is written (in the mid-size form, by the first of three launches
alone)."""
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


# a single block, the mid-size form with few and many blocks, a scan of two levels
@pytest.mark.parametrize("lg", [10, 11, 12, 16, 20, 21])
@pytest.mark.parametrize("graph", [False, True])
def test_batch_opening(pl, lg, graph):
    import torch
    n = 1 << lg
    x, z = po.uniform(n, lg), po.uniform(1, lg + 1)
    q, rem = po.div(x, po.neg(z))
    y = po.eval_(x, z)
    print("opening with the point in place", lg, graph, flush=True)
    xd = pl.to_dev(x)
    over_value = {"op": "eval_div", "lg": lg, "inp": xd, "out": torch.empty_like(xd), "z": pl.to_dev(z)}
    over_value["y"] = over_value["z"]
    out = torch.empty_like(xd)
    # the point inside the quotient's buffer, at its end
    in_quotient = {"op": "eval_div", "lg": lg, "inp": xd, "out": out, "z": out[n - 1:], "y": torch.empty_like(out[:1])}
    b = pl.Batch([over_value, in_quotient], graph=graph)
    for _ in range(2):
        over_value["z"].copy_(pl.to_dev(z))
        out.copy_(pl.to_dev(np.repeat(z, n, axis=0)))
        b.run()
        for it in (over_value, in_quotient):
            np.testing.assert_array_equal(pl.to_host(it["out"]), q)
            np.testing.assert_array_equal(pl.to_host(it["y"]), y)
    b.close()


@pytest.mark.parametrize("n", [501, 1025, 2001, 4095, 4097, 70001, (1 << 21) + 3])
def test_division_remainder(pl, n):
    x, c = po.uniform(n, n), po.uniform(1, n + 1)
    q, rem = po.div(x, c)
    print("remainder over the divisor's constant", n, flush=True)
    xd, cd = pl.to_dev(x), pl.to_dev(c)
    pl.div_linear(xd, cd, rem=cd)
    np.testing.assert_array_equal(pl.to_host(xd), q)
    np.testing.assert_array_equal(pl.to_host(cd).reshape(-1), np.asarray(rem).reshape(-1))
    xd, zd = pl.to_dev(x), pl.to_dev(c)
    pl.evaluate(xd, zd, y=zd)
    np.testing.assert_array_equal(pl.to_host(zd).reshape(-1), np.asarray(po.eval_(x, c)).reshape(-1))
