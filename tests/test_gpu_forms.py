"""Forms of the transforms and products that sizes, counts and alignment select,
each against the CPU oracle (exact residues and integers)."""
import numpy as np
import pytest

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
