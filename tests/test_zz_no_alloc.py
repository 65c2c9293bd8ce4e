"""The allocation-free solve (mbe_solve_noalloc) against mbe_solve, through
the C ABI: two calls in a row on one device, the second with a smaller
graph, then every variant, a root subset, and the size limit.

Device memory for the packed graphs comes from hipMalloc through ctypes:
the caller owns it, the library only reads it.
"""
import ctypes as C
import json
import os

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
GOLD = os.path.join(ROOT, "tests", "golden")
pytestmark = pytest.mark.gpu
M = pytest.importorskip("cumbe_amd")
import oracle_lib as O  # noqa: E402
from graphs import star_of_stars  # noqa: E402


class DevCopy:
    """A host buffer copied into device memory (hipMalloc / hipMemcpy)."""

    def __init__(self, host: np.ndarray):
        self.hip = C.CDLL("libamdhip64.so")
        self.ptr = C.c_void_p()
        assert self.hip.hipMalloc(C.byref(self.ptr), C.c_size_t(max(host.nbytes, 1))) == 0
        assert self.hip.hipMemcpy(self.ptr, host.ctypes.data_as(C.c_void_p),
                                  C.c_size_t(host.nbytes), 1) == 0  # host to device

    def close(self):
        if self.ptr:
            self.hip.hipFree(self.ptr)
            self.ptr = C.c_void_p()


def say(msg):
    print(f"[gpu] {msg}", flush=True)


def check(g, variant="cuMBE", tuning=None):
    buf, info = g.pack((tuning or {}).get("side", -1))
    dev = DevCopy(buf)
    try:
        r = M.solve_noalloc(dev.ptr.value, info, variant, tuning)
    finally:
        dev.close()
    ref = M.solve(g, variant, tuning)
    assert (r.count, r.hash) == (ref.count, ref.hash), variant
    return r


def test_noalloc_two_calls_then_smaller():
    M.init()
    gold = json.load(open(os.path.join(GOLD, "c0.json")))
    big = M.Graph.chung_lu(**gold["graph"])
    small = M.Graph.chung_lu(400, 300, 2500, 2.1, 2.1, 0, 11)
    say("noalloc: configuration 0, then a smaller graph")
    r1 = check(big)
    assert (r1.count, f"{r1.hash:#018x}") == (gold["count"], gold["hash"])
    r2 = check(small)
    assert r2.count < r1.count


def test_noalloc_variants_subset_and_limits():
    M.init()
    g = M.Graph.chung_lu(400, 300, 2500, 2.1, 2.1, 0, 11)
    for v in ("cuMBE", "noRS", "noES", "noWS"):
        say(f"noalloc variant {v}")
        check(g, v)
    say("noalloc root subset and small arenas")
    check(g, "cuMBE", {"root_begin": 3, "root_stride": 4})
    r = check(g, "cuMBE", {"arena_words": 256, "workers": 32})
    assert r.launches >= 2  # roots that did not fit ran with larger arenas
    buf, info = g.pack()
    dev = DevCopy(buf)
    try:
        with pytest.raises(M.MbeError) as e:
            M.solve_noalloc(dev.ptr.value, info, "cuMBE", {"workers": 1 << 20})
        assert e.value.status == -9
    finally:
        dev.close()


def free_bytes():
    hip = C.CDLL("libamdhip64.so")
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_list_mode_root_at_the_default_arena():
    """A hub root that list mode suits is left to a second pass, at the same
    arena size: it fits the scratch of the allocation-free solve, and a solve
    takes no larger arenas for it (they would be 48 GiB)."""
    M.init()
    n_u, n_v, off, adj = star_of_stars()
    g = M.Graph.from_csr(n_u, n_v, off, adj)
    M.solve(M.Graph.chung_lu(400, 300, 2500, 2.1, 2.1, 0, 11))
    before = free_bytes()
    say("noalloc and solve with a list-mode root")
    r = check(g, "cuMBE", {"side": 1})
    ref = O.solve(n_u, n_v, off, adj)
    assert (r.count, r.hash, r.launches) == (ref.count, ref.hash, 2)
    assert before - free_bytes() < 8 << 30


@pytest.mark.parametrize("tuning", [{"workers": 850}, {"workers": 940},
                                    {"workers": 40000, "arena_words": 512},
                                    {"workers": 60000, "arena_words": 256}], ids=str)
def test_many_workers_fit_the_scratch(tuning):
    """Explicit worker counts that the arenas, marks and rank tables leave room
    for: hand-over slots shrink, or the general engine's ring takes their place."""
    M.init()
    say(f"noalloc {tuning}")
    r = check(M.Graph.chung_lu(400, 300, 2500, 2.1, 2.1, 0, 11), "cuMBE", tuning)
    assert r.workers == tuning["workers"]
