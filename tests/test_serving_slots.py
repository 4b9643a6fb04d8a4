"""The serving loop's slots and the order of its work, on a stand-in for the
library (no GPU): streams run what is queued on them, one step per query."""
import types

import numpy as np

from cumodp_amd import serving


class _Stream:
    def __init__(self):
        self.queue = []


class _Library:
    """Streams by number; `log` holds what ran, `computing` the batches whose
    kernels are queued and have not run."""

    def __init__(self):
        self.streams, self.log, self.peak, self.live = {}, [], 0, 0

    def cumodp_stream_create(self):
        self.streams[len(self.streams) + 1] = _Stream()
        return len(self.streams)

    def cumodp_stream_destroy(self, s):
        pass

    def cumodp_dev_alloc(self, n):
        return 4096

    def cumodp_dev_free(self, p):
        return 0

    def cumodp_memcpy_h2d_async(self, dst, src, n, s):
        self.streams[s.value].queue.append("in")
        return 0

    def cumodp_two_convolution_list_dev(self, items, n, a, b, c, s):
        self.streams[s.value].queue.append(("run", n))
        self.peak = max(self.peak, sum(any(q[0] == "run" for q in t.queue)
                                       for t in self.streams.values()))
        return 0

    def cumodp_memcpy_d2h_async(self, dst, src, n, s):
        assert not any("out" in t.queue for t in self.streams.values()) or len(self.streams) == 2
        if len(self.streams) <= 2:
            assert not self.streams[s.value].queue, "the copy back follows the kernels' end"
        self.streams[s.value].queue += ["out", "out"]
        return 0

    def cumodp_stream_query(self, s):
        q = self.streams[s.value].queue
        if q:
            self.log.append((s.value, q.pop(0)))
        return 0 if q else 1


def _requests(n):
    Q = types.SimpleNamespace(n=n)
    Q.na = Q.nb = np.full(n, 100, np.int64)
    Q.nc, Q.wc, Q.bits = Q.na + Q.nb - 1, np.full(n, 3, np.int64), np.full(n, 64, np.int64)
    Q.in_off = np.arange(n + 1) * 200
    Q.out_off = np.arange(n + 1) * 199 * 3
    Q.items = np.zeros(n, serving._ITEM_DTYPE)
    Q.IN = Q.OUT = types.SimpleNamespace(ptr=1 << 20)
    return Q


def test_a_server_holds_the_slots_it_was_asked_for(monkeypatch):
    for slots in (1, 2, 3):
        lib = _Library()
        monkeypatch.setattr(serving, "lib", lambda: lib)
        srv = serving.ZmulServer(slots=slots)
        assert len(srv.slots) == slots == len(lib.streams)
        srv.close()


def test_every_batch_is_copied_back_once_and_in_order(monkeypatch):
    """One batch computes at a time with up to two slots; with more, one is
    copied back at a time."""
    for slots in (1, 2, 3):
        lib = _Library()
        monkeypatch.setattr(serving, "lib", lambda: lib)
        srv = serving.ZmulServer(slots=slots, slot_bytes=100000)
        srv._scratch_bytes = lambda bits, ny: 20000
        Q = _requests(40)
        done, stats = srv.run(Q, np.zeros(Q.n))
        assert np.isfinite(done).all() and (np.diff(done) >= 0).all()
        assert stats["batches"] >= 10
        assert lib.peak == 1 if slots <= 2 else lib.peak <= slots
        ran = [q for _, q in lib.log]
        assert ran.count("in") == stats["batches"] and ran.count("out") == 2 * stats["batches"]
        assert sum(q[1] for q in ran if q[0] == "run") == Q.n
        # with two slots, work of one batch runs between the copies of another
        outs = [i for i, (_, q) in enumerate(lib.log) if q == "out"]
        if slots <= 2:
            assert any(b - a > 1 for a, b in zip(outs[::2], outs[1::2])) == (slots == 2)
        srv.close()
