"""Transforms whose output lies over an input other than in place: from 2^7
points on the whole input is read before anything is stored, for one call and
among the items of a batch, whichever form the transform takes."""
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


# the largest one-launch sizes, the smallest of two launches; outputs ahead of and behind their input
@pytest.mark.parametrize("lg,npoly", [(7, 1), (7, 1000), (8, 1), (9, 3), (9, 400), (10, 1), (10, 100)])
@pytest.mark.parametrize("inverse", [False, True])
def test_shifted_output(pl, lg, npoly, inverse):
    import torch
    n = 1 << lg
    x = po.uniform(npoly * n, po.seed(po.OP_NTT, lg, npoly))
    ref = np.concatenate([po.ntt(x[p * n:(p + 1) * n], lg, inverse=inverse) for p in range(npoly)])
    dom = pl.Domain(lg)
    work = torch.empty((npoly * n, 4), dtype=torch.int64, device="cuda")
    for shift in (1, n // 2, n):
        for at, to in ((0, shift), (shift, 0)):
            print("shifted output", lg, npoly, inverse, at, to, flush=True)
            buf = torch.zeros((npoly * n + shift, 4), dtype=torch.int64, device="cuda")
            buf[at:at + npoly * n] = pl.to_dev(x)
            out = buf[to:to + npoly * n]
            pl.ntt_batch(buf[at:at + npoly * n], dom, npoly, inverse=inverse, out=out, work=work)
            np.testing.assert_array_equal(pl.to_host(out.clone()), ref)


@pytest.mark.parametrize("graph", [False, True])
def test_items_share_an_input(pl, graph):
    # one item in place, others of the batch read the same vector: the values from before
    import torch
    items, want, restore = [], [], []
    for lg in (7, 8, 9, 10, 12):
        for k in range(3):
            x = po.uniform(1 << lg, 16 * lg + k)
            xd = pl.to_dev(x)
            restore.append((xd, xd.clone()))
            items += [{"op": "ntt" if k else "intt", "lg": lg, "inp": xd, "out": torch.empty_like(xd)},
                      {"op": "intt" if k else "ntt", "lg": lg, "inp": xd, "out": xd},
                      {"op": "lde", "lg": lg, "lg_blowup": 1, "inp": xd,
                       "out": torch.empty((2 << lg, 4), dtype=torch.int64, device="cuda")}]
            want += [po.ntt(x, lg, inverse=not k), po.ntt(x, lg, inverse=bool(k)), po.lde(x, lg, 1, po.ref_lde_shift(1))]
    b = pl.Batch(items, graph=graph)
    for _ in range(3):
        for xd, saved in restore:
            xd.copy_(saved)
        b.run()
        for it, ref in zip(items, want):
            print("shared input", it["op"], it["lg"], graph, flush=True)
            np.testing.assert_array_equal(pl.to_host(it["out"]), ref)
    b.close()
