"""GPU tests of the launch buffers that pass from a destroyed server to the next
one: servers that need more, less or the same as the one before, with a solve
in between, all give the solve's result; and two servers at a time."""
import ctypes
import threading

import pytest

pytestmark = pytest.mark.gpu
M = pytest.importorskip("cumbe_amd")

SMALL = dict(table_cap=256, data_bytes=64 << 20, staging_bytes=16 << 20)
# workers x arena words: bigger, then smaller than what is kept, then equal
LAUNCHES = [dict(workers=64), dict(workers=300), dict(workers=16, arena_words=1 << 18),
            dict(workers=300), dict(workers=300, lds_words=600)]


def test_server_after_server():
    graphs = [M.Graph.chung_lu(300 + 40 * i, 150 + 9 * i, 1500, 2.1, 2.1, 0, i) for i in range(6)]
    want = [(r.count, r.hash) for r in (M.solve(g) for g in graphs)]

    def burst(srv):
        tickets = [srv.submit(g) for g in graphs]
        got = [srv.poll(t, wait_ms=60_000) for t in tickets]
        assert [(r.status, r.count, r.hash) for r in got] == [(0, c, h) for c, h in want]

    for tuning in LAUNCHES:
        print(f"[gpu] server {tuning}", flush=True)
        with M.Server(tuning=tuning, **SMALL) as srv:
            burst(srv)
        r = M.solve(graphs[0])
        assert (r.count, r.hash) == want[0]


def test_larger_server_beside_a_running_one():
    """A small server has left its buffers; of two larger ones the second gets
    its request first and keeps its kernel running. The first one's request
    then completes: what it needs is allocated, and nothing is freed, which
    would wait for the other's kernel."""
    g = M.Graph.chung_lu(300, 150, 1500, 2.1, 2.1, 0, 1)
    ref = M.solve(g)
    with M.Server(tuning=dict(workers=16), **SMALL) as small:
        assert small.poll(small.submit(g), wait_ms=60_000).count == ref.count
    first = M.Server(tuning=dict(workers=48), **SMALL)
    second = M.Server(tuning=dict(workers=48), **SMALL)
    got = []
    try:
        for name, srv in (("second", second), ("first", first)):
            print(f"[gpu] request to the {name} server", flush=True)
            r = srv.poll(srv.submit(g), wait_ms=20_000)
            got.append((r.count, r.hash) if r else None)
    finally:
        # at the same time: a server's end waits for the other's kernel
        ends = [threading.Thread(target=srv.close) for srv in (first, second)]
        for t in ends:
            t.start()
        for t in ends:
            t.join(60)
    assert got == [(ref.count, ref.hash)] * 2


def test_release_gives_the_buffers_back():
    """What a destroyed server keeps goes back to the device on request, and
    stays while a server is alive."""
    hip = ctypes.CDLL("libamdhip64.so")

    def free_bytes():
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    g = M.Graph.chung_lu(300, 150, 1500, 2.1, 2.1, 0, 1)
    ref = M.solve(g)
    M.release_kept()
    before = free_bytes()
    with M.Server(tuning=dict(workers=256, arena_words=1 << 20), **SMALL) as srv:
        assert srv.poll(srv.submit(g), wait_ms=60_000).count == ref.count
    assert before - free_bytes() >= 256 * 8 << 20  # the arenas
    with M.Server(tuning=dict(workers=256, arena_words=1 << 20), **SMALL) as srv:
        M.release_kept()
        assert srv.poll(srv.submit(g), wait_ms=60_000).count == ref.count
        M.release_kept()
    M.release_kept()
    assert before - free_bytes() < 64 << 20
