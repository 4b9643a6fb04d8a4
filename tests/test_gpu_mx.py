"""The matrix-core transforms against the CPU oracle, at the sizes where their
tiles, rounds and bounds change.

A transform of 2^e points runs e / 4 radix-16 rounds and one shorter round for
e mod 4, in tiles of one wave up to a workgroup; word bounds depend on the
modulus (any odd p < 2^31, with a branch of its own below 8192).  Residues are
compared exactly.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

P1, P2 = 469762049, 2013265921
TOP = 2147352577          # 2^31 - 2^17 + 1, the largest modulus bits in use: 2^17 | p - 1
SMALL = [(97, 5), (257, 8), (7681, 9), (12289, 12), (65537, 16)]


def _mul(cm, F, G, p, nout=None):
    nout = len(F) + len(G) - 1 if nout is None else nout
    dF, dG, dH = cm.DeviceArray.from_host(F), cm.DeviceArray.from_host(G), cm.DeviceArray(nout)
    cm.fftmul_uni_dev(nout - 1, dH, len(F) - 1, dF, len(G) - 1, dG, p)
    return dH.download()


@pytest.mark.parametrize("p,top", [(P1, 26), (P2, 26), (TOP, 17)] + SMALL)
def test_one_workgroup_products(cm, orc, p, top):
    rng = np.random.default_rng(p)
    for e in range(4, min(top, 13) + 1):
        n = 1 << e
        for s in (n, n - 1, n // 2 + 1):
            lf = max(1, (s + 1) * 5 // 8)
            lg = s + 1 - lf
            F = rng.integers(0, p, lf, dtype=np.int32)
            G = rng.integers(0, p, lg, dtype=np.int32)
            assert (_mul(cm, F, G, p) == orc.ntt_polymul(F, G, p)).all(), (p, e, s)
        # the largest residues, and a truncated output
        F, G = np.full(n // 2, p - 1, np.int32), np.full(n // 2, p - 1, np.int32)
        want = orc.ntt_polymul(F, G, p)
        assert (_mul(cm, F, G, p) == want).all(), (p, e)
        assert (_mul(cm, F, G, p, n // 2 + 3) == want[:n // 2 + 3]).all(), (p, e)


def test_output_over_an_operand(cm, orc):
    rng = np.random.default_rng(5)
    for e in (4, 6, 8, 11, 13):
        n = 1 << e
        F = rng.integers(0, P1, n // 2, dtype=np.int32)
        G = rng.integers(0, P1, n // 2, dtype=np.int32)
        want = orc.ntt_polymul(F, G, P1)
        buf = np.zeros(n, np.int32)
        for over in (0, 1):
            buf[:n // 2] = G if over else F
            d, other = cm.DeviceArray.from_host(buf), cm.DeviceArray.from_host(F if over else G)
            a, b = (other, d) if over else (d, other)
            cm.fftmul_uni_dev(n - 2, d, n // 2 - 1, a, n // 2 - 1, b, P1)
            assert (d.download()[:n - 1] == want).all(), (e, over)


@pytest.mark.parametrize("p,top", [(P1, 22), (P2, 21), (TOP, 17), (65537, 16)])
def test_four_step_products(cm, orc, p, top):
    """Ragged operands at odd word offsets, in the small and the large form
    (2^20 words and up), and a truncated output."""
    rng = np.random.default_rng(p + 1)
    for e in range(14, top + 1):
        n = 1 << e
        for s, off in ((n, 0), (n // 2 + 1, 1), (n - 3, 3)):
            lf = (s + 1) * 5 // 8
            lg = s + 1 - lf
            F = rng.integers(0, p, lf + off, dtype=np.int32)
            G = rng.integers(0, p, lg + off, dtype=np.int32)
            want = orc.ntt_polymul(F[off:], G[off:], p)
            dF, dG = cm.DeviceArray.from_host(F), cm.DeviceArray.from_host(G)
            for nout in (s, s // 2 + 5):
                dH = cm.DeviceArray.from_host(np.full(s + off + 8, -1, np.int32))
                cm.fftmul_uni_dev(nout - 1, dH.ptr + 4 * off, lf - 1, dF.ptr + 4 * off, lg - 1,
                                  dG.ptr + 4 * off, p)
                got = dH.download()
                assert (got[off:off + nout] == want[:nout]).all(), (p, e, s, nout)
                assert (got[:off] == -1).all() and (got[off + nout:] == -1).all(), (p, e, s, nout)


@pytest.mark.parametrize("logn", [14, 15, 17, 19, 21, 22])
def test_every_split_and_tile(cm, orc, logn):
    """Row lengths named by the tuner (columns down to 16 words) and both
    column tiles give the same words."""
    L = cm.lib()
    rng = np.random.default_rng(logn)
    n = 1 << logn
    F, G = rng.integers(0, P2, n // 2, dtype=np.int32), rng.integers(0, P2, n // 2, dtype=np.int32)
    want = orc.ntt_polymul(F, G, P2)
    keep = L.cumodp_tune_get_split(logn)
    try:
        for k2 in (12, 13, 14):
            if L.cumodp_tune_set_split(logn, k2):
                continue
            for tile in (8192, 16384):
                assert L.cumodp_tune_set_col_tile(tile) == 0
                assert (_mul(cm, F, G, P2) == want).all(), (logn, k2, tile)
    finally:
        assert L.cumodp_tune_set_split(logn, keep) == 0
        assert L.cumodp_tune_set_col_tile(16384) == 0


def test_batched_rows_of_every_size(cm, orc):
    """One batch of integer products whose rows have 2^4 .. 2^16 points in two
    and three primes (every launch of the row list), with one- and two-word
    operands, output words beyond the product's, and the most negative
    coefficients; each product against the exact schoolbook."""
    rng = np.random.default_rng(77)
    pieces, items, want, at, out = [], [], [], 0, 0
    for e in range(1, 17):
        n = 1 << e
        for bits in (1, 16, 33, 64):
            if e >= 14 and bits == 33:
                continue
            nb = int(rng.integers(1, min(n, 700)))        # short: the check is schoolbook
            na = max(1, n - nb + 1 - int(rng.integers(0, 2)))
            lim = (1 << (bits - 1)) - 1 if bits == 64 else (1 << bits) - 1
            a = rng.integers(-lim, lim, na, dtype=np.int64, endpoint=True)
            b = rng.integers(-lim, lim, nb, dtype=np.int64, endpoint=True)
            a[0], b[-1] = -lim, -lim
            if bits == 64:
                a[-1] = b[0] = -(1 << 63)
            two = bits == 33 and e % 2 == 0               # the other form, in the same call
            wc = 3 if bits == 64 else 3 + int(rng.integers(0, 3))
            words = []
            for v in (a, b):
                w = v.view(np.uint64).reshape(-1, 1)
                if two:
                    w = np.concatenate([w, np.where(v < 0, np.uint64(2**64 - 1), np.uint64(0))
                                        .reshape(-1, 1)], 1)
                words.append(np.ascontiguousarray(w).ravel())
            W = 2 if two else 1
            items.append((at, at + na * W, out, na, nb, W, W, wc, bits))
            pieces += words
            at += (na + nb) * W
            out += (na + nb - 1) * wc
            want.append((orc.zmul_i64(a, b), wc))
    arr = (cm.ZmulItem * len(items))(*[cm.ZmulItem(*t) for t in items])
    A = cm.DeviceArray.from_host(np.concatenate(pieces), np.uint64)
    H = cm.DeviceArray.from_host(np.full(out, 0x5A5A5A5A5A5A5A5A, np.uint64), np.uint64)
    assert cm.lib().cumodp_two_convolution_list_dev(arr, len(items), A.addr(), A.addr(), H.addr(),
                                                    None) == 0
    got = H.download()
    for t, (w, wc) in zip(items, want):
        r = got[t[2]:t[2] + (t[3] + t[4] - 1) * wc].reshape(-1, wc)
        assert (r[:, :3] == w).all(), t
        sign = np.where(w[:, 2] >> np.uint64(63), np.uint64(2**64 - 1), np.uint64(0))
        for j in range(3, wc):
            assert (r[:, j] == sign).all(), t


def _root(k, p):
    fac = [d for d in range(2, 1 << 16) if (p - 1) % d == 0 and all(d % q for q in range(2, d) if q * q <= d)]
    g = next(x for x in range(2, 200) if all(pow(x, (p - 1) // d, p) != 1 for d in fac))
    return pow(g, (p - 1) >> k, p)


@pytest.mark.parametrize("p,top", [(P1, 15), (P2, 15), (TOP, 15), (257, 8), (12289, 12)])
def test_row_transforms(cm, orc, p, top):
    """Rows of 2^4 .. 2^15 words (one and two launches) in the forms of few and
    of many words, with row counts that do not fill the last workgroup, at a
    4-byte aligned address."""
    rng = np.random.default_rng(p + 2)
    for k in range(4, top + 1):
        n, w = 1 << k, _root(k, p)
        for m in (1, 3, max(5, ((1 << 19) >> k) + 1)):
            X = rng.integers(0, p, m * n, dtype=np.int32)
            d = cm.DeviceArray.from_host(np.concatenate([np.full(1, 7, np.int32), X,
                                                         np.full(3, 9, np.int32)]))
            cm.cxx("list_stockham_dev_w")(d.addr(1), m, k, w, p)
            got = d.download()
            assert got[0] == 7 and (got[-3:] == 9).all(), (p, k, m)
            got = got[1:-3].reshape(m, n)
            for r in sorted({0, m // 2, m - 1}):
                assert (got[r] == orc.stockham(X[r * n:(r + 1) * n], w, p)).all(), (p, k, m, r)


@pytest.mark.parametrize("k", list(range(4, 23)))
def test_transform_and_inverse(cm, orc, k):
    p = P2 if k & 1 else P1
    rng = np.random.default_rng(k)
    n, w = 1 << k, _root(k, p)
    X = rng.integers(0, p, n, dtype=np.int32)
    Y = cm.fft_uni(X, w, p)
    assert (Y == orc.stockham(X, w, p)).all()
    assert (cm.invfft_uni(Y, w, p) == X).all()
    assert (cm.invfft_uni(X, w, p) == orc.inverse_stockham(X, w, p)).all()


@pytest.mark.parametrize("k", [23, 24, 25, 26])
def test_largest_transforms(cm, k):
    """X = a x^3 + b x^i has Y_j = a w^(3j) + b w^(ij); and back."""
    p, n = P2, 1 << k
    w, i = _root(k, P2), (1 << k) - 12345
    X = np.zeros(n, np.int32)
    X[3], X[i] = 123456789, 987654321
    Y = cm.fft_uni(X, w, p)
    for j in (0, 1, 2, 5, 16, 255, 4096, n // 2 + 1, n - 1, 0x155555 % n):
        want = (123456789 * pow(w, 3 * j, p) + 987654321 * pow(w, i * j, p)) % p
        assert int(Y[j]) == want, (k, j)
    assert (cm.invfft_uni(Y, w, p) == X).all()


@pytest.mark.parametrize("p,top", [(P1, 15), (P2, 15), (12289, 12), (65537, 14)])
def test_tree_levels_with_wrapped_leading_terms(cm, orc, p, top):
    """Levels above 8 multiply whole monic nodes on exactly their length: the
    leading term wraps onto the constant one.  Zero, equal and largest points
    make constant terms 0 and p - 1."""
    for k in range(9, top + 1):
        rng = np.random.default_rng(k)
        for pts in (rng.integers(0, p, 1 << k, dtype=np.int32), np.zeros(1 << k, np.int32),
                    np.full(1 << k, p - 1, np.int32)):
            tree = cm.subproduct_tree(pts, p)
            lev = tree[k - 1]
            want = orc.ntt_polymul(lev[0], lev[1], p) if (1 << k) < p - 1 else None
            for i in range(9, k + 1):
                a, b = tree[i - 1][-2], tree[i - 1][-1]
                assert int(tree[i][-1][-1]) == 1
                low = orc.plain_polymul(a[:40], b[:40], p)[:40]
                assert (tree[i][-1][:40] == low).all(), (p, k, i)
                high = orc.plain_polymul(a[::-1][:40].copy(), b[::-1][:40].copy(), p)[:40]
                assert (tree[i][-1][::-1][:40] == high).all(), (p, k, i)
            x = int(pts[1])
            assert int(orc.poly_eval(tree[k][0], np.array([x], np.int32), p)[0]) == 0
            if want is not None and p % (1 << (k + 1)) == 1:
                assert (tree[k][0] == want).all(), (p, k)


@pytest.mark.parametrize("p,ks", [(P1, (8, 9, 10, 11, 12, 13, 14, 15, 18)), (P2, (9, 13, 14)),
                                  (TOP, (9, 16, 17)), (12289, (10, 11, 12))])
def test_transposed_evaluation(cm, orc, p, ks):
    """Values by the transposed algorithm (k >= 9 with 2^(k+1) | p - 1) against
    the remainder tree, which runs when the remainders are kept, and Horner's
    rule on a sample; coefficients are any 32-bit words."""
    rng = np.random.default_rng(p + 3)
    for k in ks:
        n = 1 << k
        pts = rng.integers(0, p, n, dtype=np.int32)
        pts[0], pts[-1], pts[n // 2] = 0, p - 1, pts[1]
        F = rng.integers(0, 1 << 32, n, dtype=np.uint64)
        F[:3] = (1 << 32) - 1
        got = cm.fast_evaluation(F.astype(np.uint32).view(np.int32), pts, p)
        Fp = (F % p).astype(np.int32)
        if k <= 14:
            r = cm.eval_steps("fastEvaluation", pts, p, Fp, flag=1)
            assert (got == np.concatenate([r["fL"][1], r["fR"][1]])).all(), (p, k)
        idx = np.unique(np.concatenate([[0, 1, n // 2, n - 1], rng.integers(0, n, 60)]))
        assert (got[idx] == orc.poly_eval(Fp, pts[idx], p)).all(), (p, k)


@pytest.mark.parametrize("p", [P1, P2])
def test_list_products_in_pieces(cm, orc, p):
    """List products above 2^13 points run modulo 2, 3 or 4 factors x^8192 - omega,
    or 8192 + 4096 points up to 12288 words; in one task each when the list is
    long and one task per factor when it is short.  The operands' chunks of
    8192 words are folded, so one side is also taken shorter and longer than
    that."""
    rng = np.random.default_rng(p + 4)
    words = (8193, 12287, 12288, 12289, 16384, 16385, 24576, 24577, 32768)
    shapes = [(s, lf) for s in words for lf in (s // 2, s - 40, 41)]
    F, G, want, items, fo, go = [], [], [], [], 0, 0
    for s, lf in shapes:
        lg = s + 1 - lf
        f, g = (rng.integers(0, p, n, dtype=np.int32) for n in (lf, lg))
        f[:2], g[:2] = p - 1, p - 1
        items.append((fo, go, lf - 1, lg - 1))
        F.append(f), G.append(g), want.append(orc.ntt_polymul(f, g, p))
        fo, go = fo + lf, go + lg
    dF = cm.DeviceArray.from_host(np.concatenate(F))
    dG = cm.DeviceArray.from_host(np.concatenate(G))
    for copies in (1, 40):
        n = len(items) * copies
        arr, ho = (cm.MulItem * n)(), 0
        for i in range(n):
            x = arr[i]
            x.f_off, x.g_off, x.df, x.dg = items[i % len(items)]
            x.h_off = ho
            ho += x.df + x.dg + 1
        H = cm.DeviceArray.from_host(np.full(ho, -1, np.int32))
        cm.list_fftmul_dev(arr, dF, dG, H, p)
        got = H.download()
        for i in range(n):
            w = want[i % len(items)]
            assert (got[arr[i].h_off:arr[i].h_off + len(w)] == w).all(), (i, shapes[i % len(items)])


@pytest.mark.parametrize("p", [P1, P2])
def test_columns_of_many_tiles(cm, p):
    """From 512 column tiles on, one workgroup per CU takes several tiles if the
    operands end on a whole quad of words: the same products as with tiles of
    half the width, which run one workgroup per tile."""
    L = cm.lib()
    rng = np.random.default_rng(p + 5)
    for e, shapes in ((22, ((0, 0, 0), (4, 4, 0), (-4, 8, 3), (2, 2, 0), (0, 1, 1))),
                      (23, ((0, 0, 0), (1, 0, 5))), (24, ((0, -8, 0), (0, 0, 1)))):
        for da, db, cut in shapes:
            lf, lg = (5 << (e - 3)) - da, (3 << (e - 3)) - db - (da == db == 0)
            lf, lg = (lf, lg & ~3) if da % 4 == 0 and db % 4 == 0 else (lf, lg)
            F, G = (rng.integers(0, p, n, dtype=np.int32) for n in (lf, lg))
            nout = lf + lg - 1 - cut
            old = L.cumodp_tune_get_col_tile()
            got = _mul(cm, F, G, p, nout)
            try:
                assert L.cumodp_tune_set_col_tile(8192) == 0
                want = _mul(cm, F, G, p, nout)
            finally:
                L.cumodp_tune_set_col_tile(old)
            assert (got == want).all(), (e, lf, lg, nout)
