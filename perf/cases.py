"""Performance cases of the prover operators: the calls a PLONK prover makes
through plffi (the binding of include/pl.h), over the sizes it makes them at.

A case is a dict with a "kind" and its sizes:

  ntt    npoly transforms of 2^lg elements, forward or inverse (pl_ntt,
         pl_ntt_batch)
  lde    2^lg coefficients to blowup * 2^lg evaluations (pl_lde; blowup 3 or a
         power of two)
  coset  transform over the coset 7<w>, forward or inverse (pl_coset_ntt)
  perm   permutation grand product z over 2^lg rows, fused, or as the ratio
         vector followed by its prefix product (pl_perm_grand_product;
         pl_perm_ratio + pl_grand_product)
  open   a polynomial of n coefficients opened at a point: its value and the
         quotient by (X - zeta) (pl_eval + pl_div_linear)
  vec    element-wise operator over n elements (pl_vec_op)
  batch  the uneven polynomials of one proof planned once, replayed per proof
         (pl_batch_create, pl_batch_run)

A field element is 32 bytes, four int64 words of a canonical Montgomery
residue; results are exact integers.  Domains, workspaces, output buffers and
batch plans are what a prover keeps between proofs, so `prepare` makes them.
Domains use the library's default pass splits.
"""
import os
import random
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ppopp26-artifact_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import plffi  # noqa: E402

R = 0x73EDA753299D7D483339D80809A1D80553BDA402FFFE5BFEFFFFFFFF00000001
MONT = (1 << 256) % R
R_INV = pow(MONT, R - 2, R)
TOP = R >> 192  # a top word below this keeps the element below R
MULMOD = 2 * 128  # operations of a product: 2 * 8^2 multiply-adds of 32-bit limbs


def listed():
    return [
        # the smallest transform of a proof (lookup and public-input columns): launches and latency
        {"name": "ntt_2p10", "kind": "ntt", "lg": 10, "npoly": 1, "inverse": False},
        # one witness column of a small circuit, evaluations to coefficients
        {"name": "intt_2p16", "kind": "ntt", "lg": 16, "npoly": 1, "inverse": True},
        # the headline transform
        {"name": "ntt_2p24", "kind": "ntt", "lg": 24, "npoly": 1, "inverse": False},
        # the largest circuit's column
        {"name": "intt_2p26", "kind": "ntt", "lg": 26, "npoly": 1, "inverse": True},
        # an odd number of mid-size columns transformed in one call
        {"name": "intt_13x2p15", "kind": "ntt", "lg": 15, "npoly": 13, "inverse": True},
        # a column extended by 4, the ordinary commitment of a mid-size circuit
        {"name": "lde4_2p20", "kind": "lde", "lg": 20, "blowup": 4},
        # a column extended by 8, a large circuit
        {"name": "lde8_2p22", "kind": "lde", "lg": 22, "blowup": 8},
        # the quotient polynomial back to coefficients from its coset evaluations
        {"name": "icoset_2p18", "kind": "coset", "lg": 18, "inverse": True},
        # the permutation argument of a 2^20-row circuit
        {"name": "perm_2p20", "kind": "perm", "lg": 20, "fused": True},
        # the same with the ratio kept (a lookup argument needs it), 2^21 rows
        {"name": "ratio_gp_2p21", "kind": "perm", "lg": 21, "fused": False},
        # a blinded polynomial (a few coefficients above 2^20) opened at the challenge
        {"name": "open_2p20_5", "kind": "open", "n": (1 << 20) + 5},
        # one proof: 56 polynomials of 2^12 .. 2^20, 35 NTTs, 14 extensions by 4, 7 openings
        {"name": "proof_batch", "kind": "batch", "polys": 56, "lg_lo": 12, "lg_hi": 20, "mix": 1},
    ]


def _log_between(rng, lo, hi):
    """An odd whole number spread over the logarithm of [lo, hi]."""
    return int(lo * (hi / lo) ** rng.random()) | 1


def draw(rng):
    kind = rng.choice(["ntt", "ntt", "ntt", "lde", "lde", "coset", "perm", "open", "open", "vec", "batch"])
    if kind == "ntt":
        lg = rng.randint(8, 25)
        npoly = 1 if rng.random() < 0.5 else rng.randint(2, max(2, min(40, 1 << max(0, 24 - lg))))
        return {"kind": "ntt", "lg": lg, "npoly": npoly, "inverse": rng.random() < 0.5}
    if kind == "lde":
        blowup = rng.choice([2, 3, 4, 8, 16])
        return {"kind": "lde", "lg": rng.randint(8, 21 if blowup == 16 else 22), "blowup": blowup}
    if kind == "coset":
        return {"kind": "coset", "lg": rng.randint(8, 24), "inverse": rng.random() < 0.5}
    if kind == "perm":
        return {"kind": "perm", "lg": rng.randint(10, 23), "fused": rng.random() < 0.6}
    if kind == "open":
        return {"kind": "open", "n": _log_between(rng, 500, 1 << 24)}
    if kind == "vec":
        return {"kind": "vec", "op": rng.choice(["mul", "inv", "div", "add"]), "n": _log_between(rng, 1000, 1 << 23)}
    lo = rng.randint(10, 14)
    return {"kind": "batch", "polys": rng.randint(12, 56), "lg_lo": lo, "lg_hi": rng.randint(lo + 2, 20),
            "mix": rng.randrange(1 << 20)}


def _elements(n, seed, salt=0):
    """n uniform canonical elements on the GPU, shape (n, 4)."""
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 1000003 + salt) & 0x7FFFFFFFFFFFFFFF)
    x = torch.randint(-(1 << 63), (1 << 63) - 1, (n, 4), dtype=torch.int64, device="cuda", generator=g)
    x[:, 3] = torch.randint(0, TOP, (n,), dtype=torch.int64, device="cuda", generator=g)
    return x


def _empty(n):
    return torch.empty((n, 4), dtype=torch.int64, device="cuda")


def _host(v):
    """A number as a (1, 4) array of its Montgomery words."""
    m = v * MONT % R
    return np.array([[(m >> (64 * i)) & 0xFFFFFFFFFFFFFFFF for i in range(4)]], dtype=np.uint64)


def _polys(case):
    """[(op, lg)] of a proof: 5 of 8 transforms, 2 of 8 extensions, 1 of 8 openings."""
    rng = random.Random(case["mix"])
    n = case["polys"]
    ops = ["eval_div"] * max(1, n // 8) + ["lde"] * max(1, n // 4)
    ops += ["ntt"] * (n - len(ops))
    rng.shuffle(ops)
    return [(op, rng.randint(case["lg_lo"], case["lg_hi"])) for op in ops]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "ntt":
        lg, npoly = case["lg"], case["npoly"]
        return {"kind": kind, "x": _elements(npoly << lg, seed), "npoly": npoly, "inverse": case["inverse"],
                "dom": plffi.Domain(lg), "out": _empty(npoly << lg), "work": _empty(npoly << lg)}
    if kind == "lde":
        b = case["blowup"]
        dom = plffi.LdeDomain(case["lg"], 0, blowup3=True) if b == 3 else plffi.LdeDomain(case["lg"], b.bit_length() - 1)
        return {"kind": kind, "x": _elements(1 << case["lg"], seed), "dom": dom, "out": _empty(b << case["lg"]),
                "work": _empty(dom.work_bytes // 32)}
    if kind == "coset":
        n = 1 << case["lg"]
        return {"kind": kind, "x": _elements(n, seed), "dom": plffi.CosetDomain(case["lg"]), "out": _empty(n),
                "work": _empty(n), "inverse": case["inverse"]}
    if kind == "perm":
        lg = case["lg"]
        n = 1 << lg
        return {"kind": kind, "w": [_elements(n, seed, j) for j in range(3)],
                "s": [_elements(n, seed, 3 + j) for j in range(3)], "beta": _elements(1, seed, 6),
                "gamma": _elements(1, seed, 7), "k": np.concatenate([_host(1), _host(7), _host(13)]),
                "dom": plffi.Domain(lg), "out": _empty(n), "fused": case["fused"],
                "work": torch.empty(plffi.lib().pl_vec_work_bytes(n), dtype=torch.uint8, device="cuda")}
    if kind == "open":
        n = case["n"]
        zeta = _elements(1, seed, 1)
        return {"kind": kind, "x": _elements(n, seed), "zeta": zeta, "c": plffi.vec_op("neg", zeta), "q": _empty(n),
                "y": _empty(1), "work": torch.empty(plffi.lib().pl_scan_work_bytes(n), dtype=torch.uint8, device="cuda")}
    if kind == "vec":
        n = case["n"]
        return {"kind": kind, "op": case["op"], "a": _elements(n, seed), "b": _elements(n, seed, 1), "out": _empty(n),
                "work": torch.empty(plffi.lib().pl_vec_work_bytes(n), dtype=torch.uint8, device="cuda")}
    items, outs = [], []
    for i, (op, lg) in enumerate(_polys(case)):
        n = 1 << lg
        it = {"op": op, "lg": lg, "inp": _elements(n, seed, 2 * i), "out": _empty(4 * n if op == "lde" else n)}
        if op == "lde":
            it["lg_blowup"] = 2
        outs.append(it["out"])
        if op == "eval_div":
            it["z"], it["y"] = _elements(1, seed, 2 * i + 1), _empty(1)
            outs.append(it["y"])
        items.append(it)
    return {"kind": kind, "batch": plffi.Batch(items), "outs": outs}


def run(state):
    kind = state["kind"]
    if kind == "ntt":
        if state["npoly"] == 1:
            return plffi.ntt(state["x"], state["dom"], inverse=state["inverse"], out=state["out"], work=state["work"])
        return plffi.ntt_batch(state["x"], state["dom"], state["npoly"], inverse=state["inverse"], out=state["out"],
                               work=state["work"])
    if kind == "lde":
        return plffi.lde(state["x"], state["dom"], out=state["out"], work=state["work"])
    if kind == "coset":
        return plffi.coset_ntt(state["x"], state["dom"], inverse=state["inverse"], out=state["out"], work=state["work"])
    if kind == "perm":
        z = plffi.perm_ratio(state["w"], state["s"], state["beta"], state["gamma"], state["k"], state["dom"],
                             out=state["out"], grand_product=state["fused"], work=state["work"])
        return z if state["fused"] else plffi.grand_product(z, work=state["work"])
    if kind == "open":
        y = plffi.evaluate(state["x"], state["zeta"], y=state["y"], work=state["work"])
        state["q"].copy_(state["x"])  # the division is in place and the prover keeps the polynomial
        return y, plffi.div_linear(state["q"], state["c"], work=state["work"])
    if kind == "vec":
        b = state["b"] if state["op"] in ("mul", "div", "add") else None
        return plffi.vec_op(state["op"], state["a"], b, out=state["out"], work=state["work"])
    state["batch"].run()
    return state["outs"]


def _work_of(kind, lg=0, n=0, blowup=1):
    """(elements moved, products) of one operator."""
    if kind == "ntt":
        return 2 * n, n // 2 * lg
    if kind == "lde":
        return n + blowup * n, blowup * (n // 2 * lg + n)
    if kind == "open":
        return 2 * n, 2 * n  # value and quotient from the same Horner recurrence, with its split
    raise ValueError(kind)


def work(case):
    kind = case["kind"]
    if kind == "ntt":
        n = 1 << case["lg"]
        el, mul = [case["npoly"] * v for v in _work_of("ntt", case["lg"], n)]
    elif kind == "lde":
        el, mul = _work_of("lde", case["lg"], 1 << case["lg"], case["blowup"])
    elif kind == "coset":
        n = 1 << case["lg"]
        el, mul = 2 * n, n // 2 * case["lg"] + n
    elif kind == "perm":
        n = 1 << case["lg"]
        # six columns in, one out; three products per row in the terms, four in
        # the products of three, three in the batch inversion, two in the scan
        el, mul = 7 * n, 12 * n
    elif kind == "open":
        el, mul = _work_of("open", n=case["n"])
    elif kind == "vec":
        two = case["op"] in ("mul", "div", "add")
        el = (3 if two else 2) * case["n"]
        mul = {"mul": 1, "add": 0, "inv": 3, "div": 4}[case["op"]] * case["n"]
    else:
        el = mul = 0
        for op, lg in _polys(case):
            a, b = _work_of("open" if op == "eval_div" else op, lg, 1 << lg, 4)
            el, mul = el + a, mul + b
    return {"bytes": 32 * el, "flops": MULMOD * mul}


def _ints(t):
    w = t.cpu().numpy().view(np.uint64).astype(object)
    return [int(a) | int(b) << 64 | int(c) << 128 | int(d) << 192 for a, b, c, d in w]


def _tensor(v):
    a = np.array([[(x >> (64 * i)) & 0xFFFFFFFFFFFFFFFF for i in range(4)] for x in v], dtype=np.uint64)
    return torch.from_numpy(a.view(np.int64))


def _dft(x, w):
    if len(x) == 1:
        return x
    e, o = _dft(x[::2], w * w % R), _dft(x[1::2], w * w % R)
    t, c = [], 1
    for v in o:
        t.append(v * c % R)
        c = c * w % R
    return [(a + b) % R for a, b in zip(e, t)] + [(a - b) % R for a, b in zip(e, t)]


def exact(case, seed):
    """The result in Python's whole numbers, where that is quick."""
    if case["kind"] == "ntt" and case["npoly"] << case["lg"] <= 1 << 17:
        lg, n = case["lg"], 1 << case["lg"]
        w = pow(7, (R - 1) >> lg, R)
        x = _ints(_elements(case["npoly"] << lg, seed))
        out = []
        for p in range(case["npoly"]):
            y = _dft(x[p * n:(p + 1) * n], pow(w, R - 2, R) if case["inverse"] else w)
            f = pow(n, R - 2, R) if case["inverse"] else 1
            out += [v * f % R for v in y]
        return _tensor(out)
    if case["kind"] == "open" and case["n"] <= 1 << 21:
        x, z = _ints(_elements(case["n"], seed)), _ints(_elements(1, seed, 1))[0] * R_INV % R
        q, acc = [0] * len(x), 0
        for i in range(len(x) - 1, -1, -1):
            q[i] = acc
            acc = (acc * z + x[i]) % R
        return _tensor([acc]), _tensor(q)
    if case["kind"] == "vec" and case["n"] <= 1 << 19:
        a = _ints(_elements(case["n"], seed))
        b = _ints(_elements(case["n"], seed, 1))
        if case["op"] == "add":
            return _tensor([(x + y) % R for x, y in zip(a, b)])
        if case["op"] == "mul":
            return _tensor([x * y * R_INV % R for x, y in zip(a, b)])
    return None
