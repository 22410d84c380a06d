"""Planned steps on bit rows (the workgroup kernels) and tasks with a vertex per lane (the
wavefront kernel) against the oracle at the sizes where words, chunks, planes and lanes end: condensed graphs of 31 to 129 vertices (32 ids a word), tasks of
one to a few chunks of 32 steps, member counts beyond the bit planes (14) and least clique
sizes on either side of them. Also: lists that no bit row can stand for are walked."""
import ctypes
import os
import random

import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def cluster_graph(seed, sizes, density, links):
    """Disjoint near-complete clusters with a few arcs between them: adjacency lists."""
    rng = random.Random(seed)
    n = sum(sizes)
    out = [set() for _ in range(n)]
    at = 0
    for size in sizes:
        for u in range(at, at + size):
            for v in range(at, at + size):
                if u != v and rng.random() < density:
                    out[u].add(v)
        at += size
    for _ in range(links):
        u, v = rng.randrange(n), rng.randrange(n)
        if u != v:
            out[u].add(v)
    return [sorted(x) for x in out]


def write(path, out):
    with open(path, "w") as f:
        for row in out:
            f.write(" ".join(map(str, row)) + "\n")


CASES = [  # cluster sizes, density, links, gammas, least size
    ([31], 0.82, 0, 0.85, 0.85, 16), ([32], 0.82, 0, 0.85, 0.85, 16), ([33], 0.82, 0, 0.85, 0.85, 17),
    ([20, 11], 0.92, 20, 0.85, 0.85, 9), ([20, 12], 0.92, 30, 0.85, 0.85, 9), ([22, 22, 20], 0.92, 60, 0.85, 0.9, 10),
    ([22, 22, 21], 0.92, 60, 0.9, 0.85, 10), ([24, 24, 24, 24, 1], 0.88, 120, 0.8, 0.8, 15),
    ([26, 26, 26, 26, 24], 0.9, 200, 0.85, 0.85, 16), ([26, 26, 26, 26, 25], 0.9, 200, 0.85, 0.85, 17),
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_planned_steps_match_oracle(dqc, tmp_path, case):
    sizes, density, links, go, gi, mn = CASES[case]
    path = str(tmp_path / "g.txt")
    write(path, cluster_graph(100 + case, sizes, density, links))
    ref = str(tmp_path / "ref.max")
    count, st = orc.run(path, go, gi, mn, None, ref, threads=2)
    want = open(ref, "rb").read() if os.path.exists(ref) else b""
    for wave, schedule, split in ((-1, dqc.SCHED_FIFO, 0), (-1, dqc.SCHED_SIZE, 2), (256, dqc.SCHED_FIFO, 0)):
        cfg = dqc.Config()
        cfg.host_addfail_check = 1
        cfg.wave_tasks, cfg.schedule = wave, schedule
        cfg.split_branches, cfg.split_chunk = (split, 3) if split else (0, 0)
        got_path = str(tmp_path / f"got_{wave}_{schedule}.max")
        got, gst = dqc.search_file(path, go, gi, mn, None, got_path, cfg)
        data = open(got_path, "rb").read() if os.path.exists(got_path) else b""
        assert (got, gst.tasks_expanded, gst.branches, gst.raw_cliques) == (count, st.tasks, st.branches, st.raw_cliques)
        assert data == want
    # two copies in one batch: the level-0 tasks (31 to 129 vertices, on either side of the 64
    # lanes) run as ordinary tasks, small ones with a vertex per lane, their results buffered
    for resident in (0, 3):
        cfg = dqc.Config()
        cfg.host_addfail_check = 1
        cfg.resident_steps = resident
        files = [str(tmp_path / f"batch{resident}_{i}.max") for i in range(2)]
        counts, bst = dqc.search_batch([path, path], go, gi, mn, files, cfg)
        assert counts == [count, count]
        assert (bst.tasks_expanded, bst.branches, bst.raw_cliques) == (2 * st.tasks, 2 * st.branches, 2 * st.raw_cliques)
        assert all((open(f, "rb").read() if os.path.exists(f) else b"") == want for f in files)


def run_uploaded(dqc, lists, records, mn, gamma):
    """The level-0 task of an uploaded graph, run to completion; counts and sorted cliques."""
    n = len(lists[0])
    arrays = [dqc._csr_arrays(x) for x in lists]
    length = 2 * (max(n, mn) + 2) + 2
    md = (ctypes.c_int32 * length)(*dqc.min_degrees(gamma, length - 1))
    ub = (ctypes.c_int32 * length)(*[int(d / gamma) for d in range(length)])
    cfg = dqc.Config()
    cfg.host_addfail_check = 1
    cfg.wave_tasks = -1
    with dqc.Engine(cfg) as eng:
        lib = eng.lib
        eng._check(lib.dqc_upload_graph(eng.h, ctypes.c_int32(n), *[a for pair in arrays for a in pair]), "upload")
        eng._check(lib.dqc_set_tables(eng.h, md, md, ub, ub, ctypes.c_int32(length), ctypes.c_int32(mn)), "tables")
        eng.push_task(records, 0, 0, 0)
        eng.run(dqc.SCHED_FIFO)
        st = eng.stats()
        return st.tasks_expanded, st.branches, sorted(tuple(sorted(c)) for c in eng.cliques())


def test_lists_without_bit_rows(dqc):
    """Two-hop lists in descending order have no bit row of the same meaning: the kernels walk
    them, with the result of the ascending lists (a list is a set here)."""
    out = cluster_graph(7, [20, 14], 0.93, 0)
    n = len(out)
    inn = [[u for u in range(n) if v in out[u]] for v in range(n)]
    two = [[x for x in (range(20) if v < 20 else range(20, n)) if x != v] for v in range(n)]
    records = [(v, 0, len(out[v]), 0, len(inn[v]), len(two[v])) for v in range(n)]
    want = run_uploaded(dqc, (out, inn, two), records, 8, 0.85)
    assert want[2]
    assert run_uploaded(dqc, (out, inn, [x[::-1] for x in two]), records, 8, 0.85) == want
