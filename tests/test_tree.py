"""The tree engine at the edges of its tiers: levels just inside and just
outside a tile (64 candidates in P, 128 in Q, rows of 1, 2, 4, 8 and more
words), wide levels, and hand-over between workers, against the oracle -- on
the CPU under the wave64 emulator and, marked gpu, on the device.

The graphs are windows: row i is adjacent to the columns i*s .. i*s + d - 1;
a few rows in the middle have a hole. All rows have about the same degree, so a row's P are the
windows before it and its Q those after it, up to d / s of each.
"""
import os
import random
import re
import subprocess
import time

import pytest

import oracle_lib as O
from graphs import csr_from_edges, star_of_stars

M = pytest.importorskip("cumbe_amd")
EMU_DIR = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emu")

# (rows, window, step, rows with a hole): P up to window / step - 1 and as many Q
CASES = [
    (9, 1, 1, 0), (70, 63, 1, 0), (140, 64, 1, 3), (140, 65, 1, 3), (140, 66, 1, 3),
    (170, 67, 1, 4), (180, 129, 1, 0), (180, 130, 1, 2), (40, 128, 8, 4), (40, 129, 4, 4),
    (90, 256, 4, 2), (90, 257, 4, 2), (40, 512, 16, 4), (40, 513, 16, 4), (24, 1100, 64, 4),
]


def windows(n, d, s, holes):
    gone = {n // 2 + i: i * s + d // 2 - i for i in range(holes)}
    edges = [(i, i * s + j) for i in range(n) for j in range(d) if gone.get(i) != j]
    return csr_from_edges(n, (n - 1) * s + d, edges)


# (rows, columns, columns per row): universes of 10, 66 and 130 words below
# which L' is a few bits, each in a word of its own
SCATTERED = [(18, 5000, 600), (9, 40000, 4200), (8, 60000, 8300)]


def scattered(n, cols, d):
    rng = random.Random(n)
    return csr_from_edges(n, cols, [(i, j) for i in range(n) for j in rng.sample(range(cols), d)])


def case_id(c):
    return "-".join(map(str, c))


@pytest.fixture(scope="module")
def emu():
    subprocess.run(["make", "-C", EMU_DIR], check=True, capture_output=True)

    def run(*args):
        out = subprocess.run([os.path.join(EMU_DIR, "emu_run"), *map(str, args)],
                             capture_output=True, text=True, timeout=300)
        assert out.returncode == 0, out.stderr
        m = re.search(r"count (\d+) hash (0x[0-9a-f]+) nodes (\d+) donated (\d+) stolen (\d+)",
                      out.stdout)
        return [int(x, 0) for x in m.groups()]
    return run


@pytest.mark.parametrize("case", CASES, ids=case_id)
def test_tiles_emulated(case, emu, tmp_path):
    """Default budget; frames and rows in the arena (no LDS room) with
    hand-over at every step."""
    g = windows(*case)
    ref = O.solve(*g)
    path = str(tmp_path / "w.bi")
    M.Graph.from_csr(*g).write_bi(path)
    for opts in (("-w", 4), ("-w", 8, "-l", 420, "-i", 1, "-S", 0)):
        count, h, nodes, donated, stolen = emu(*opts, "bi", path)
        assert (count, h) == (ref.count, ref.hash), opts
        assert donated == stolen and nodes >= count


@pytest.mark.parametrize("case", SCATTERED, ids=case_id)
def test_scattered_levels_emulated(case, emu, tmp_path):
    g = scattered(*case)
    ref = O.solve(*g)
    path = str(tmp_path / "s.bi")
    M.Graph.from_csr(*g).write_bi(path)
    for opts in (("-w", 4), ("-w", 8, "-l", 420, "-i", 1)):
        count, h, _, donated, stolen = emu(*opts, "-S", 0, "bi", path)
        assert (count, h) == (ref.count, ref.hash), opts
        assert donated == stolen


@pytest.mark.gpu
@pytest.mark.parametrize("case", SCATTERED, ids=case_id)
def test_scattered_levels_on_gpu(case):
    g = scattered(*case)
    ref = O.solve(*g)
    gg = M.Graph.from_csr(*g)
    for t in ({"side": 0}, {"side": 0, "workers": 24, "donate_interval": 1, "lds_words": 420}):
        print(f"scattered {case} tuning {t}", flush=True)
        r = M.solve(gg, "cuMBE", t)
        assert (r.count, r.hash) == (ref.count, ref.hash), t


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=case_id)
def test_tiles_on_gpu(case):
    g = windows(*case)
    ref = O.solve(*g)
    gg = M.Graph.from_csr(*g)
    for t in ({}, {"side": 0, "workers": 24, "donate_interval": 1}, {"side": 0, "lds_words": 420}):
        print(f"windows {case} tuning {t}", flush=True)
        r = M.solve(gg, "cuMBE", t or None)
        assert (r.count, r.hash) == (ref.count, ref.hash), t


PLANTED = (6500, 1900, 0.008, 60, 8, 40, 0.05, 3)


@pytest.mark.parametrize("workers", [2, 4])
def test_late_count_keeps_idle_workers(workers, emu):
    """One deep root, and atomics without a result performed up to 20 ms late:
    a worker that finds no root must not send the others away while the one
    with the root has not been counted yet. Levels handed to a worker that
    has left would be missing from the count."""
    ref = O.solve_roots(*M.Graph.er_planted(*PLANTED).csr(), begin=11, end=12, threads=1)
    for seed in range(1, 7):
        count, h, _, donated, stolen = emu("-w", workers, "-i", 1, "-b", 11, "-e", 12, "-D", 20000,
                                           "-G", seed, "er", *PLANTED)
        assert (count, h) == (ref.count, ref.hash), seed
        assert donated == stolen > 0


def serve_emu(*args):
    subprocess.run(["make", "-C", EMU_DIR], check=True, capture_output=True)
    return subprocess.run([os.path.join(EMU_DIR, "emu_run"), *map(str, args)], capture_output=True,
                          text=True, timeout=300)


def test_served_node_budget_stops_busy_workers():
    """A serving kernel's node budget stops workers that never idle: the only
    worker, with 14 roots of a request before it, reports a part of it."""
    out = serve_emu("-w", 1, "-S", 1, "-n", 500, "serve", "e120,14,0.7,0,0,0,0,1")
    assert int(re.search(r"nodes (\d+)", out.stdout).group(1)) < 2000, out.stdout + out.stderr


def test_handed_level_needs_no_descriptor():
    """A serving kernel's descriptors are written while it runs, and a worker
    that takes a handed-over level may hold an older copy of their cache lines:
    with the descriptor changed once all roots are claimed, the hash stays."""
    spec = (300, 18, 0.6, 0, 0, 0, 0, 1)
    ref = O.solve(*M.Graph.er_planted(*spec).csr())
    out = serve_emu("-w", 8, "-i", 1, "-S", 1, "-Z", 1000, "serve", "e" + ",".join(map(str, spec)))
    assert out.returncode == 0, out.stderr + out.stdout
    assert f"count {ref.count} hash {ref.hash:#018x} err 0 done 1" in out.stdout
    assert int(re.search(r"stolen (\d+)", out.stdout).group(1)) > 0


@pytest.mark.parametrize("opts", [(), ("-t", 0)], ids=["tree", "general"])
def test_time_limit_without_donation(opts):
    """The abort flag is seen within a task whatever the donation interval: a
    root that takes many seconds here ends soon after the limit of 0.2 s."""
    subprocess.run(["make", "-C", EMU_DIR], check=True, capture_output=True)
    t0 = time.time()
    out = subprocess.run([os.path.join(EMU_DIR, "emu_run"), "-w", "2", "-b", "16", "-e", "17", "-i",
                          "4000000000", "-A", "200", *map(str, opts), "er", *map(str, PLANTED)],
                         capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and " aborted\n" in out.stdout, out.stderr + out.stdout
    assert time.time() - t0 < 15
    assert int(re.search(r"count (\d+)", out.stdout).group(1)) < 1 << 16


def test_node_budget_counts_nodes(emu, tmp_path):
    """The node budget is in nodes of the tree as they are reported, on wide
    levels too (some 300 candidates a root here): a budget that covers them
    does not stop the solve, a quarter of it does."""
    g = scattered(600, 800, 8)
    ref = O.solve(*g)
    path = str(tmp_path / "sparse.bi")
    M.Graph.from_csr(*g).write_bi(path)
    nodes = emu("-w", 4, "-S", 0, "bi", path)[2]
    count, h, *_ = emu("-w", 4, "-S", 0, "-n", nodes + 1, "bi", path)
    assert (count, h) == (ref.count, ref.hash)
    assert emu("-w", 4, "-S", 0, "-n", nodes // 4, "bi", path)[0] < ref.count


def test_list_mode_root_keeps_the_arena_size(tmp_path):
    """A root that the tree engine leaves to list mode fits the arenas that
    there are: its pass does not ask for larger ones."""
    g = star_of_stars()
    ref = O.solve(*g)
    path = str(tmp_path / "star.bi")
    M.Graph.from_csr(*g).write_bi(path)
    out = serve_emu("-p", 8, "-a", 32768, "-S", 1, "bi", path).stdout
    assert out.startswith(f"count {ref.count} hash {ref.hash:#018x}")
    assert "launches 2" in out and "arena 32768" in out
