"""GPU test of the launch buffers that pass from a destroyed server to the next
one: servers that need more, less or the same as the one before, with a solve
in between, all give the solve's result."""
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
