"""What the library is measured on: one dict per call that its users make.

Every case goes through a public entry point with the operands already where
that entry point takes them: device buffers for the `_dev` calls, host arrays
for the drop-in `cumodp_fftmul_uni`.  Twiddle tables and scratch belong to the
library and are built by its first call of a size, as in a user's process.

Kinds:
  mul    one product mod p on device buffers (cumodp_fftmul_uni_dev)
  host   one product mod p on host arrays (cumodp_fftmul_uni, modpn's call)
  list   many products of uneven degree (cumodp_list_fftmul_dev)
  ntt    one natural-order transform in place (stockham_dev, inverse_stockham_dev)
  rows   the same transform of many rows in place (list_stockham_dev)
  zmul   one exact integer product (cumodp_two_convolution_poly_mul_dev)
  zlist  a batch of integer products (cumodp_two_convolution_list_dev), as one
         batch of the serving loop holds them
  tree   the subproduct tree over 2^k points (cumodp_subproduct_tree_dev)
  eval   a polynomial of degree < 2^k at 2^k points (cumodp_fast_evaluation_dev)

Outputs are whole numbers (residues mod p, integer words) with one right value
each, so there is no exact(): they are compared word for word.
"""
import ctypes as C
import math
import random

import numpy as np
import torch

import cumodp_amd as cm

P1 = cm.P1   # 469762049 = 7 2^26 + 1, below 2^30
P2 = cm.P2   # 2013265921 = 15 2^27 + 1, above 2^30
BITS = (16, 32, 48, 64)


def listed():
    return [
        # the smallest call in use: a 2048-point product, launch and latency bound
        {"name": "mul_2048", "kind": "mul", "df": 1023, "dg": 1023, "p": P1},
        # an ordinary product of two polynomials of unlike, odd lengths
        {"name": "mul_ragged", "kind": "mul", "df": 70000, "dg": 30010, "p": P1},
        # the headline: 2^24 points modulo a prime above 2^30
        {"name": "mul_2e24", "kind": "mul", "df": (1 << 23) - 1, "dg": (1 << 23) - 1, "p": P2},
        # the drop-in call on host arrays, copies included
        {"name": "host_2e17", "kind": "host", "df": 65535, "dg": 65535, "p": P1},
        # a batch of uneven pairs
        {"name": "list_4096", "kind": "list", "count": 4096, "lo": 32, "hi": 16384, "p": P1},
        # stand-alone transforms, both directions, and many short rows
        {"name": "ntt_2e20", "kind": "ntt", "k": 20, "inverse": False, "p": P2},
        {"name": "ntt_inv_2e16", "kind": "ntt", "k": 16, "inverse": True, "p": P1},
        {"name": "rows_2e11", "kind": "rows", "m": 2000, "k": 11, "p": P1},
        # an exact integer product of coefficients in (-10^10, 10^10)
        {"name": "zmul_16384", "kind": "zmul", "na": 16384, "nb": 16384, "bits": 34},
        # one batch of integer requests of mixed degree and width
        {"name": "zlist_96", "kind": "zlist", "count": 96, "lo": 64, "hi": 65536},
        # the subproduct tree and the evaluation on it
        {"name": "tree_2e16", "kind": "tree", "k": 16, "p": P1},
        {"name": "eval_2e16", "kind": "eval", "k": 16, "p": P1},
    ]


def _log(rng, lo, hi):
    """a whole number in [lo, hi], its logarithm uniform"""
    return min(hi, int(lo * (hi / lo) ** rng.random() + rng.random()))


def draw(rng):
    kind = rng.choice(("mul", "mul", "mul", "host", "list", "list", "ntt", "rows", "zmul", "zlist",
                       "tree", "eval"))
    p = rng.choice((P1, P2))
    if kind in ("mul", "host"):
        df = _log(rng, 128, (1 << 23) - 1 if kind == "mul" else 1 << 18)
        return {"kind": kind, "df": df, "dg": _log(rng, max(128, df // 16), df), "p": p}
    if kind == "list":
        hi = _log(rng, 512, 50000)
        # the largest list holds about the words of the listed one
        most = max(16, min(4096, 20000000 // hi))
        return {"kind": kind, "count": _log(rng, 16, most), "lo": 32, "hi": hi, "p": p}
    if kind == "ntt":
        return {"kind": kind, "k": rng.randint(12, 22), "inverse": rng.random() < 0.5, "p": p}
    if kind == "rows":
        k = rng.randint(6, 15)
        return {"kind": kind, "m": _log(rng, 3, (1 << 22) >> k), "k": k, "p": p}
    if kind == "zmul":
        na = _log(rng, 64, 65536)
        return {"kind": kind, "na": na, "nb": _log(rng, max(64, na // 16), na),
                "bits": rng.choice(BITS)}
    if kind == "zlist":
        return {"kind": kind, "count": _log(rng, 4, 96), "lo": 64, "hi": _log(rng, 1024, 65536)}
    return {"kind": kind, "k": rng.randint(6, 15), "p": p}


# ---- inputs ------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _residues(gen, n, p):
    return torch.randint(0, p, (n,), generator=gen, device="cuda", dtype=torch.int32)


def _signed(gen, n, bits):
    """n int64 coefficients of at most `bits` bits, sign included for 64"""
    if bits == 64:
        return torch.randint(-(1 << 63), (1 << 63) - 1, (n,), generator=gen, device="cuda",
                             dtype=torch.int64)
    top = (1 << bits) - 1
    return torch.randint(-top, top + 1, (n,), generator=gen, device="cuda", dtype=torch.int64)


class _Buf:
    """A device tensor as the bindings take their device arrays."""

    def __init__(self, t):
        self.t = t

    def addr(self):
        return C.c_void_p(self.t.data_ptr())


def _root(k, p):
    """a root of unity of order 2^k mod p: 3 or 31 generates the units"""
    g = {P1: 3, P2: 31}[p]
    return pow(g, (p - 1) >> k, p)


def _degrees(case, n):
    """2 n degrees, log-uniform in [lo, hi]; the layout belongs to the case, so
    passes of other seeds do the same amount of work"""
    rng = random.Random("%d %d %d" % (case["count"], case["lo"], case["hi"]))
    return [_log(rng, case["lo"], case["hi"]) for _ in range(2 * n)]


def _words_out(bits, na, nb):
    lg = max(0, math.ceil(math.log2(min(na, nb)))) if min(na, nb) > 1 else 0
    return (2 * bits + lg + 1 + 63) // 64


def _out(n, dtype=torch.int32):
    return torch.zeros(n, dtype=dtype, device="cuda")


def _zitems(case):
    """the items of one batch, packed as the serving loop packs them, and the
    input and output words they take"""
    n = case["count"]
    deg = _degrees(case, n)
    rng = random.Random("bits %d %d" % (n, case["hi"]))
    items = (cm.ZmulItem * n)()
    at = out = 0
    for i in range(n):
        na, nb, bits = deg[i] + 1, deg[n + i] + 1, rng.choice(BITS)
        wc = _words_out(bits, na, nb)
        it = items[i]
        it.a_off, it.b_off, it.c_off, it.na, it.nb = at, at + na, out, na, nb
        it.wa = it.wb = 1
        it.wc, it.bits = wc, bits
        at += na + nb
        out += (na + nb - 1) * wc
    return items, at, out


def prepare(case, seed):
    kind, gen = case["kind"], _gen(seed)
    s = {"case": case}
    if kind == "host":
        rng = np.random.default_rng(seed)
        s["F"] = rng.integers(0, case["p"], case["df"] + 1, dtype=np.int32)
        s["G"] = rng.integers(0, case["p"], case["dg"] + 1, dtype=np.int32)
    elif kind == "mul":
        s["F"] = _residues(gen, case["df"] + 1, case["p"])
        s["G"] = _residues(gen, case["dg"] + 1, case["p"])
        s["H"] = _out(case["df"] + case["dg"] + 1)
    elif kind == "list":
        deg = _degrees(case, case["count"])
        items, nf, ng, nh = cm.make_items(deg[:case["count"]], deg[case["count"]:])
        s["items"] = items
        s["F"], s["G"] = _Buf(_residues(gen, nf, case["p"])), _Buf(_residues(gen, ng, case["p"]))
        s["H"] = _Buf(_out(nh))
    elif kind in ("ntt", "rows"):
        s["X"] = _residues(gen, case.get("m", 1) << case["k"], case["p"])
        s["w"] = _root(case["k"], case["p"])
    elif kind == "zmul":
        s["A"], s["B"] = _signed(gen, case["na"], case["bits"]), _signed(gen, case["nb"], case["bits"])
        s["wc"] = _words_out(case["bits"], case["na"], case["nb"])
        s["H"] = _out((case["na"] + case["nb"] - 1) * s["wc"], torch.int64)
    elif kind == "zlist":
        s["items"], n_in, n_out = _zitems(case)
        # the coefficients of item i, one draw of 64 bits each cut to its width
        x = _signed(gen, n_in, 64)
        width = np.repeat([it.bits for it in s["items"]], [it.na + it.nb for it in s["items"]])
        shift = torch.from_numpy(64 - width).to("cuda")
        s["A"] = x >> shift
        s["H"] = _out(n_out, torch.int64)
    elif kind == "tree":
        s["points"] = _residues(gen, 1 << case["k"], case["p"])
        s["H"] = _out(cm.lib().cumodp_subproduct_tree_words(case["k"]))
    else:
        s["points"] = _residues(gen, 1 << case["k"], case["p"])
        s["F"] = _residues(gen, 1 << case["k"], case["p"])
        s["H"] = _out(1 << case["k"])
    return s


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def _ok(status):
    if status:
        raise RuntimeError("status 0x%x: %s" % (status, cm.lib().cumodp_last_error().decode()))


# ---- one pass ----------------------------------------------------------------
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "mul":
        df, dg = case["df"], case["dg"]
        cm.fftmul_uni_dev(df + dg, s["H"].data_ptr(), df, s["F"].data_ptr(), dg,
                          s["G"].data_ptr(), case["p"])
        return s["H"]
    if kind == "host":
        return cm.poly_mul(s["F"], s["G"], case["p"])
    if kind == "list":
        cm.list_fftmul_dev(s["items"], s["F"], s["G"], s["H"], case["p"])
        return s["H"].t
    if kind == "ntt":
        name = "inverse_stockham_dev_w" if case["inverse"] else "stockham_dev_w"
        cm.cxx(name)(_ptr(s["X"]), 1 << case["k"], case["k"], s["w"], case["p"])
        return s["X"]
    if kind == "rows":
        cm.cxx("list_stockham_dev_w")(_ptr(s["X"]), case["m"], case["k"], s["w"], case["p"])
        return s["X"]
    if kind == "zmul":
        _ok(cm.lib().cumodp_two_convolution_poly_mul_dev(
            _ptr(s["A"]), case["na"], 1, _ptr(s["B"]), case["nb"], 1, _ptr(s["H"]), s["wc"],
            case["bits"], None))
        return s["H"]
    if kind == "zlist":
        _ok(cm.lib().cumodp_two_convolution_list_dev(
            s["items"], len(s["items"]), _ptr(s["A"]), _ptr(s["A"]), _ptr(s["H"]), None))
        return s["H"]
    if kind == "tree":
        _ok(cm.lib().cumodp_subproduct_tree_dev(_ptr(s["points"]), case["k"], case["p"],
                                                _ptr(s["H"]), None))
        return s["H"]
    _ok(cm.lib().cumodp_fast_evaluation_dev(_ptr(s["F"]), _ptr(s["points"]), case["k"], case["p"],
                                            _ptr(s["H"]), None))
    return s["H"]


# ---- what a pass cannot do without -------------------------------------------
def _product(lf, lg):
    """words and operations of one product mod p: operands in, product out;
    three transforms of the product's own length (no padding), ten
    instructions per radix-2 butterfly"""
    n = lf + lg - 1
    return 4 * (lf + lg + n), 10 * 1.5 * n * math.log2(max(n, 2))


def _zproduct(na, nb, bits):
    """one integer product of one-word coefficients: words in and out; its
    2 K y-products modulo two or three primes, K limbs a coefficient"""
    plan = cm.two_convolution_plan(bits, na, nb)
    nprimes, limbs = plan[0], plan[1]
    nbytes = 8 * (na + nb + (na + nb - 1) * _words_out(bits, na, nb))
    return nbytes, nprimes * 2 * limbs * _product(na, nb)[1]


def work(case):
    kind = case["kind"]
    if kind in ("mul", "host"):
        parts = [_product(case["df"] + 1, case["dg"] + 1)]
    elif kind == "list":
        n = case["count"]
        d = _degrees(case, n)
        parts = [_product(d[i] + 1, d[n + i] + 1) for i in range(n)]
    elif kind in ("ntt", "rows"):
        n = case.get("m", 1) << case["k"]
        parts = [(8 * n, 10 * 0.5 * n * case["k"])]
    elif kind == "zmul":
        parts = [_zproduct(case["na"], case["nb"], case["bits"])]
    elif kind == "zlist":
        parts = [_zproduct(it.na, it.nb, it.bits) for it in _zitems(case)[0]]
    else:
        k = case["k"]
        # one product per node of each level; the evaluation divides twice on
        # the way down (two products of the node's size)
        level = [((1 << (k - i)), _product(1 << (i - 1), 1 << (i - 1))[1]) for i in range(1, k + 1)]
        flops = sum(n * f for n, f in level)
        if kind == "tree":
            parts = [(4 * ((1 << k) + cm.lib().cumodp_subproduct_tree_words(k)), flops)]
        else:
            parts = [(12 << k, 3 * flops)]
    return {"bytes": sum(b for b, _ in parts), "flops": sum(f for _, f in parts)}
