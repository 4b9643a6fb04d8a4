"""The list multiply's task words against the CPU oracle (exact residues)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

P1, P2 = 469762049, 2013265921


def _list(cm, F, G, p):
    """The products of the operand pairs, one call."""
    df, dg = [len(f) - 1 for f in F], [len(g) - 1 for g in G]
    items, nf, ng, nh = cm.make_items(df, dg)
    H = cm.DeviceArray.from_host(np.full(nh + 4, -1, np.int32))
    cm.list_fftmul_dev(items, cm.DeviceArray.from_host(np.concatenate(F)),
                       cm.DeviceArray.from_host(np.concatenate(G)), H, p)
    got = H.download()
    assert (got[nh:] == -1).all()
    return [got[it.h_off:it.h_off + it.df + it.dg + 1] for it in items]


def test_schoolbook_products_of_many_tasks(cm, orc):
    """The output count of a task word goes up to the largest product: 2^20 words
    are 512 tasks, among products of one task and of a transform."""
    rng = np.random.default_rng(3)
    F = [rng.integers(0, P2, n, dtype=np.int32) for n in (5, (1 << 20) + 3, 31, 3000, 1, 2047)]
    G = [rng.integers(0, P2, n, dtype=np.int32) for n in ((1 << 20) + 2, 2, 2018, 3000, 1, 2)]
    for f, g, h in zip(F, G, _list(cm, F, G, P2)):
        if min(len(f), len(g)) > 100:
            assert (h == orc.ntt_polymul(f, g, P2)).all(), (len(f), len(g))
        else:
            assert (h == orc.plain_polymul(f, g, P2)).all(), (len(f), len(g))
