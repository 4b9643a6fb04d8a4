"""The list multiply's task words and its two task sizes, against the CPU oracle.

Tasks have 512 threads and 8192 words or 1024 threads and 16384 words, by what the
products of 2^14 and 2^15 points fill; residues are compared exactly.
"""
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


def _sized(rng, p, words):
    """Operands of products of the given lengths, one side up to three times the
    other, with the largest residues at their ends."""
    F, G = [], []
    for s in words:
        lf = int(rng.integers(s // 4, 3 * s // 4 + 1))
        f, g = (rng.integers(0, p, n, dtype=np.int32) for n in (lf, s + 1 - lf))
        f[0] = f[-1] = g[0] = g[-1] = p - 1
        F.append(f), G.append(g)
    return F, G


# lengths of the products of a list, by the form it takes (256 CUs)
LISTS = {
    # large tasks in one round: tiles of every size, halves of 2^15-point products
    "large": [16384] * 100 + [8193] * 20 + [16385, 24576, 24577, 32768] * 3 +
             [8192, 4097, 2048, 1025, 512, 200, 100] * 3,
    # large tasks in several rounds
    "rounds": [16000] * 240 + [32000] * 20 + [5000] * 9,
    # small tasks, every piece a task although there are 1024 tasks and more
    "pieces": [8000] * 1010 + [32768, 24577, 24576, 16385, 16384, 12289, 12288] * 3,
}


@pytest.mark.parametrize("p", [P1, P2])
@pytest.mark.parametrize("form", sorted(LISTS))
def test_lists_of_both_task_sizes(cm, orc, p, form):
    rng = np.random.default_rng(7)
    words = LISTS[form]
    F, G = _sized(rng, p, words)
    got = _list(cm, F, G, p)
    seen = {}
    for f, g, h, s in zip(F, G, got, words):
        seen[s] = seen.get(s, 0) + 1
        if seen[s] <= 3 or seen[s] % 50 == 0:
            assert (h == orc.ntt_polymul(f, g, p)).all(), (form, s, len(f))


def test_large_tasks_in_a_graph(cm, orc):
    """Captured after an eager call, replayed with eager calls in between."""
    import ctypes as C
    L = cm.lib()
    rng = np.random.default_rng(8)
    F, G = _sized(rng, P1, [16384] * 128 + [30000] * 6)
    df, dg = [len(f) - 1 for f in F], [len(g) - 1 for g in G]
    items, nf, ng, nh = cm.make_items(df, dg)
    swapped = cm.make_items(dg, df)[0]
    dF, dG = (cm.DeviceArray.from_host(np.concatenate(x)) for x in (F, G))
    H = cm.DeviceArray(nh)
    st = L.cumodp_stream_create()
    try:
        cm.list_fftmul_dev(items, dF, dG, H, P1, st)
        assert L.cumodp_stream_synchronize(C.c_void_p(st)) == 0
        want = H.download()
        for i in (0, 127, 128, 133):
            it = items[i]
            assert (want[it.h_off:it.h_off + it.df + it.dg + 1] ==
                    orc.ntt_polymul(F[i], G[i], P1)).all(), i
        assert L.cumodp_graph_begin(C.c_void_p(st)) == 0
        cm.list_fftmul_dev(items, dF, dG, H, P1, st)
        graph = L.cumodp_graph_end(C.c_void_p(st))
        assert graph
        other = cm.DeviceArray(nh)
        for _ in range(3):
            H.upload(np.full(nh, -1, np.int32))
            assert L.cumodp_graph_launch(C.c_void_p(graph), C.c_void_p(st)) == 0
            cm.list_fftmul_dev(swapped, dG, dF, other, P1, st)   # the same scratch
            assert L.cumodp_stream_synchronize(C.c_void_p(st)) == 0
            assert (H.download() == want).all() and (other.download() == want).all()
        assert L.cumodp_graph_destroy(C.c_void_p(graph)) == 0
    finally:
        L.cumodp_stream_destroy(C.c_void_p(st))
