"""Forms of the transforms and products that sizes, counts and alignment select,
each against the CPU oracle (exact residues and integers)."""
import numpy as np
import pytest

from cumodp_amd.serving import out_words

pytestmark = pytest.mark.gpu

P1, P2 = 469762049, 2013265921


def _root(k, p):
    return pow({P1: 3, P2: 31}[p], (p - 1) >> k, p)


def _rows(cm, orc, m, k, p, off, check, seed):
    """m rows of 2^k words `off` words into an allocation; the rows of `check`
    against the oracle, the words around them unchanged."""
    n, w = 1 << k, _root(k, p)
    X = np.random.default_rng(seed).integers(0, p, m * n, dtype=np.int32)
    d = cm.DeviceArray.from_host(np.concatenate([np.full(off, 7, np.int32), X,
                                                 np.full(5, 9, np.int32)]))
    cm.cxx("list_stockham_dev_w")(d.addr(off), m, k, w, p)
    got = d.download()
    assert (got[:off] == 7).all() and (got[-5:] == 9).all(), (k, m, off)
    for r in check:
        at = off + r * n
        assert (got[at:at + n] == orc.stockham(X[r * n:(r + 1) * n], w, p)).all(), (k, m, off, r)


@pytest.mark.parametrize("p", [P1, P2])
@pytest.mark.parametrize("k", [4, 5, 6, 7, 8])
def test_many_short_rows(cm, orc, k, p):
    """From 2^19 words on, a tile of 1024 words is loaded and stored in quads; row
    counts around a whole tile, at each alignment."""
    base = (1 << 19) >> k
    per = max(1, 1024 >> k)
    for off, m in enumerate((base, base + 1, base + per - 1, base + per + 1)):
        check = sorted({0, 1, per - 1, per, m // 2, m - 2, m - 1})
        _rows(cm, orc, m, k, p, off, check, 100 * k + off)


class _Splits:
    """Named row lengths {k: k2} for a while."""

    def __init__(self, cm, named):
        self.L, self.named = cm.lib(), named

    def __enter__(self):
        self.keep = {k: self.L.cumodp_tune_get_split(k) for k in self.named}
        for k, k2 in self.named.items():
            assert self.L.cumodp_tune_set_split(k, k2) == 0, (k, k2)
            assert self.L.cumodp_tune_get_split(k) == k2

    def __exit__(self, *exc):
        for k, k2 in self.keep.items():
            assert self.L.cumodp_tune_set_split(k, k2) == 0
            assert self.L.cumodp_tune_get_split(k) == k2


@pytest.mark.parametrize("k2", [12, 13, 14])
def test_a_named_split_is_the_one_that_runs(cm, k2):
    """The tables of a split are built by its first product, and the
    non-allocating multiply refuses a split without tables."""
    k, n = 18, 1 << 18
    rng = np.random.default_rng(k2)
    F, G = (cm.DeviceArray.from_host(rng.integers(0, P1, n // 2, dtype=np.int32)) for _ in "FG")
    H = cm.DeviceArray(n - 1)
    def mul(**kw):
        cm.fftmul_uni_dev(n - 2, H, n // 2 - 1, F, n // 2 - 1, G, P1, **kw)
        return H.download()
    want = mul()
    assert (mul(noalloc=True) == want).all()
    assert cm.lib().cumodp_tune_get_split(k) not in (12, 13, 14)
    with _Splits(cm, {k: k2}):
        with pytest.raises(cm.CumodpError):
            mul(noalloc=True)
        assert (mul() == want).all()
        assert (mul(noalloc=True) == want).all()


def test_splits_refused(cm):
    L = cm.lib()
    for k, k2 in ((13, 12), (14, 11), (14, 14), (17, 9), (20, 11), (26, 12), (27, 14), (22, 15)):
        keep = L.cumodp_tune_get_split(k)
        assert L.cumodp_tune_set_split(k, k2) == cm.CUMODP_ASSUMPTION_ERROR, (k, k2)
        assert L.cumodp_tune_get_split(k) == keep


@pytest.mark.parametrize("k,k2", [(24, 12), (25, 12), (25, 13), (26, 13)])
def test_longest_columns(cm, k, k2):
    """Columns of 2^12 and 2^13 words in both tiles, against the library's own split
    and the product's values at 1, -1 and the square roots of -1."""
    L, p, n = cm.lib(), P2, 1 << k
    rng = np.random.default_rng(k)
    F, G = (rng.integers(0, p, m, dtype=np.int32) for m in (n // 2 - 3, n // 2 + 1))
    dF, dG, dH = cm.DeviceArray.from_host(F), cm.DeviceArray.from_host(G), cm.DeviceArray(n - 3)

    def mul():
        cm.fftmul_uni_dev(n - 4, dH, len(F) - 1, dF, len(G) - 1, dG, p)
        return dH.download()

    def at(X):
        """values at the fourth roots of unity"""
        s = [int(X[j::4].astype(np.int64).sum()) for j in range(4)]
        return [sum(v * pow(w, j, p) for j, v in enumerate(s)) % p
                for w in (pow(31, (p - 1) // 4 * t, p) for t in range(4))]

    want = mul()
    assert [a * b % p for a, b in zip(at(F), at(G))] == at(want)
    try:
        with _Splits(cm, {k: k2}):
            for tile in (16384, 8192):
                assert L.cumodp_tune_set_col_tile(tile) == 0
                assert (mul() == want).all(), (k, k2, tile)
    finally:
        assert L.cumodp_tune_set_col_tile(16384) == 0


@pytest.mark.parametrize("named", [{14: 13, 15: 13, 16: 13, 17: 14}, {14: 12, 15: 12, 16: 14, 17: 12},
                                   {14: 13, 15: 14, 16: 12, 17: 13}])
@pytest.mark.parametrize("p", [P1, P2])
def test_trees_and_lists_on_named_splits(cm, orc, p, named):
    """Monic nodes, middle products (with coefficients of any 32 bits) and batched
    products over columns of 2 to 32 words: the words of the library's own
    splits."""
    rng = np.random.default_rng(9)
    k = 16
    pts = rng.integers(0, p, 1 << k, dtype=np.int32)
    pts[:2] = 0, p - 1
    F = rng.integers(0, 1 << 32, 1 << k, dtype=np.uint64).astype(np.uint32).view(np.int32)
    f = [rng.integers(0, p, m, dtype=np.int32) for m in (30000, 40000, 70001, 33000)]
    items, nf, ng, nh = cm.make_items([len(x) - 1 for x in f], [len(x) - 2 for x in f])
    dF = cm.DeviceArray.from_host(np.concatenate(f))
    dG = cm.DeviceArray.from_host(np.concatenate([x[::-1][1:] for x in f]))

    def run():
        H = cm.DeviceArray.from_host(np.full(nh, -1, np.int32))
        cm.list_fftmul_dev(items, dF, dG, H, p)
        tree = cm.subproduct_tree(pts, p)
        return [H.download(), cm.fast_evaluation(F, pts, p)] + [np.concatenate(t) for t in tree]

    want = run()
    it = items[2]
    assert (want[0][it.h_off:it.h_off + it.df + it.dg + 1] ==
            orc.ntt_polymul(f[2], f[2][::-1][1:].copy(), p)).all()
    with _Splits(cm, named):
        for a, b in zip(run(), want):
            assert (a == b).all()


@pytest.mark.parametrize("e", [13, 14, 17, 21])
def test_cyclic_product_at_any_word(cm, orc, e):
    """stockham_poly_mul_dev on operands at every word of a 16-byte block."""
    p, n = P1, 1 << e
    rng = np.random.default_rng(e)
    F, G = (rng.integers(0, p, n, dtype=np.int32) for _ in "FG")
    full = np.append(orc.ntt_polymul(F, G, p), 0).astype(np.int64)
    want = ((full[:n] + full[n:]) % p).astype(np.int32)
    for a, b in ((0, 0), (1, 0), (0, 2), (3, 3)):
        dF = cm.DeviceArray.from_host(np.concatenate([np.full(a, 5, np.int32), F, [6] * 4]).astype(np.int32))
        dG = cm.DeviceArray.from_host(np.concatenate([np.full(b, 5, np.int32), G, [6] * 4]).astype(np.int32))
        cm.cxx("stockham_poly_mul_dev")(n, e, dF.addr(a), dG.addr(b), p)
        got, other = dF.download(), dG.download()
        assert (got[a:a + n] == want).all(), (e, a, b)
        assert (got[:a] == 5).all() and (got[a + n:] == 6).all(), (e, a, b)
        assert (other[:b] == 5).all() and (other[b + n:] == 6).all(), (e, a, b)


def test_more_rows_than_a_grid_holds(cm, orc):
    """65540 rows of 2^14 words: both passes are launched in parts."""
    k, m, p = 14, 65540, P1
    n, w = 1 << k, _root(k, P1)
    d = cm.DeviceArray(m * n)
    cm.cxx("reset_vector_dev")(m * n, d.addr())
    rng = np.random.default_rng(14)
    rows = {r: rng.integers(0, p, n, dtype=np.int32) for r in (0, 1, 65534, 65535, 65536, m - 1)}
    for r, x in rows.items():
        d.upload(x, r * n)
    cm.cxx("list_stockham_dev_w")(d.addr(), m, k, w, p)
    for r, x in rows.items():
        assert (d.download(n, r * n) == orc.stockham(x, w, p)).all(), r
    for r in (2, 65533, 65537):
        assert (d.download(n, r * n) == 0).all(), r
    d.free()


@pytest.mark.parametrize("m,k", [(9, 17), (5, 18), (3, 19), (3, 20), (2, 21), (2, 22), (70, 14), (40, 15),
                                 (17, 16), (300, 14)])
@pytest.mark.parametrize("p", [P1, P2])
def test_rows_of_two_passes(cm, orc, m, k, p):
    """Several rows above 2^13 words, more than 2^20 words in all: row tiles of 8
    and 16 frequencies; with the inverse root and 1/2^k, back again."""
    n, w = 1 << k, _root(k, p)
    _rows(cm, orc, m, k, p, 1, sorted({0, m // 2, m - 1}), 10 * k + m)
    X = np.random.default_rng(k).integers(0, p, m * n, dtype=np.int32)
    d = cm.DeviceArray.from_host(X)
    f = cm.cxx("list_stockham_dev_w")
    f(d.addr(), m, k, w, p)
    f(d.addr(), m, k, pow(w, p - 2, p), p)
    back = d.download().astype(np.int64) * pow(n, p - 2, p) % p
    assert (back == X).all()


@pytest.mark.parametrize("persistent,count,logn", [(1, 70, 16), (1, 35, 17), (1, 20, 18), (1, 9, 19),
                                                   (0, 100, 14), (0, 300, 14), (0, 150, 15),
                                                   (0, 40, 15)])
@pytest.mark.parametrize("p", [P1, P2])
def test_batched_four_step_products(cm, orc, persistent, count, logn, p):
    """Lists of one four-step size above 2^20 and above 2^22 words: two and four
    sets per lane in rows of 2^8 to 2^11 words."""
    rng = np.random.default_rng(count)
    n, df, dg = 1 << logn, [], []
    for _ in range(count):
        s = int(rng.integers(n // 2 + 1, n + 1))
        x = int(rng.integers(s // 4, s // 2))
        df.append(x)
        dg.append(s - 1 - x)
    items, nf, ng, nh = cm.make_items(df, dg)
    F, G = (rng.integers(0, p, m, dtype=np.int32) for m in (nf, ng))
    H = cm.DeviceArray.from_host(np.full(nh, -1, np.int32))
    L = cm.lib()
    keep = L.cumodp_tune_get_list_persistent()
    try:
        assert L.cumodp_tune_set_list_persistent(persistent) == 0
        cm.list_fftmul_dev(items, cm.DeviceArray.from_host(F), cm.DeviceArray.from_host(G), H, p)
        got = H.download()
    finally:
        assert L.cumodp_tune_set_list_persistent(keep) == 0
    for i in sorted({0, 1, count // 2, count - 1}):
        it = items[i]
        f, g = F[it.f_off:it.f_off + it.df + 1], G[it.g_off:it.g_off + it.dg + 1]
        assert (got[it.h_off:it.h_off + it.df + it.dg + 1] == orc.ntt_polymul(f, g, p)).all(), i


def _zpair(rng, s, nb, bits):
    """Operands of s + 1 coefficients in all, the extremes of the width among them."""
    lim = (1 << (bits - 1)) - 1 if bits == 64 else (1 << bits) - 1
    a, b = (rng.integers(-lim, lim, n, dtype=np.int64, endpoint=True) for n in (s + 1 - nb, nb))
    a[0] = a[-1] = b[0] = -lim
    return a, b


def test_integer_batch_of_long_rows(cm, orc):
    """One batch with rows of 2^17 to 2^21 points (and short ones): four-step passes
    of several column and row lengths in one list, and the rows above 2^20 after
    it.  One operand is short, since the check is schoolbook."""
    rng = np.random.default_rng(21)
    A, items, at, out = [], [], 0, 0
    for e in (17, 21, 19, 20, 18, 5, 13, 17, 20):
        for bits in (16, 34, 64) if e < 20 else (34,):
            s = (1 << e) - int(rng.integers(0, 3))
            a, b = _zpair(rng, s, int(rng.integers(5, 24)), bits)
            if len(items) % 2:
                a, b = b, a
            wc = out_words(bits, len(a), len(b))
            items.append((at, at + len(a), out, len(a), len(b), 1, 1, wc, bits))
            A += [a, b]
            at += len(a) + len(b)
            out += (len(a) + len(b) - 1) * wc
    arr = (cm.ZmulItem * len(items))(*[cm.ZmulItem(*t) for t in items])
    D = cm.DeviceArray.from_host(np.concatenate(A).view(np.uint64), np.uint64)
    H = cm.DeviceArray.from_host(np.full(out, 0x5A5A5A5A5A5A5A5A, np.uint64), np.uint64)
    assert cm.lib().cumodp_two_convolution_list_dev(arr, len(items), D.addr(), D.addr(), H.addr(),
                                                    None) == 0
    got = H.download()
    for i, t in enumerate(items):
        na, nb, wc = t[3], t[4], t[7]
        want = orc.zmul_i64(A[2 * i], A[2 * i + 1])[:, :wc]
        assert (got[t[2]:t[2] + (na + nb - 1) * wc].reshape(-1, wc) == want).all(), t


@pytest.mark.parametrize("e,bits", [(18, 16), (19, 34), (19, 64), (20, 34), (21, 34), (21, 64)])
def test_long_integer_products(cm, orc, e, bits):
    rng = np.random.default_rng(e)
    a, b = _zpair(rng, (1 << e) - 1, 19, bits)
    wc = out_words(bits, len(a), len(b))
    dA, dB = (cm.DeviceArray.from_host(x.view(np.uint64), np.uint64) for x in (a, b))
    H = cm.DeviceArray((len(a) + len(b) - 1) * wc, np.uint64)
    assert cm.lib().cumodp_two_convolution_poly_mul_dev(
        dA.addr(), len(a), 1, dB.addr(), len(b), 1, H.addr(), wc, bits, None) == 0
    assert (H.download().reshape(-1, wc) == orc.zmul_i64(a, b)[:, :wc]).all()


@pytest.mark.parametrize("e,p", [(22, P1), (22, P2), (23, P2)])
def test_column_loop(cm, orc, e, p):
    """512 column tiles and more, operands of whole quads and unlike lengths, the
    product whole and cut inside a quad."""
    rng = np.random.default_rng(e)
    lf, lg = (5 << (e - 3)) - 12, (3 << (e - 3)) - 8
    F, G = (rng.integers(0, p, m, dtype=np.int32) for m in (lf, lg))
    want = orc.ntt_polymul(F, G, p)
    dF, dG = cm.DeviceArray.from_host(F), cm.DeviceArray.from_host(G)
    for nout in (lf + lg - 1, lf + 1):
        H = cm.DeviceArray.from_host(np.full(lf + lg + 3, -1, np.int32))
        cm.fftmul_uni_dev(nout - 1, H, lf - 1, dF, lg - 1, dG, p)
        got = H.download()
        assert (got[:nout] == want[:nout]).all() and (got[nout:] == -1).all(), nout
