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
