"""The work whose time is measured: what users of the enumerator have it do, on seeded inputs.

Kinds of cases (the key "kind" of a case):

  search   one whole search of a small graph file, from the text file to the maximal file
           (what the command line does);
  enum     the complete enumeration of one prepared graph on an open handle;
  batch    the complete enumeration of a batch of small graphs on one handle, and the
           maximal-set files of all of them;
  window   a window of level-0 branches of a graph too large to enumerate, and the depth-1
           tasks they produce (a first look at a large graph, or a shard of it);
  tasks    one expansion batch of given depth-1 tasks: their children and cliques;
  unit     a bounded unit of a large graph: a window of level-0 branches and their subtrees
           down to a depth, under one of the schedules;
  serve    one allocation-free expansion of a task, everything in the caller's device
           memory (code that may not allocate: serving loops, graph capture);
  predict  the cost model's predictions for a set of tasks;
  train    training of the cost model from a task log.

Graphs are the two families of the synthetic workloads: Erdos-Renyi and R-MAT, each with
planted quasi-cliques. The result of a handle comes in an order that depends on the
scheduling of the device, so run() puts sets and tasks into one fixed order, as a program
that compares or stores them does.
"""
import ctypes
import math
import os
import tempfile

import numpy as np
import torch

import cudqc_amd as dq
from cudqc_amd import learn

DEVICE = "cuda:0"
SCHEDULES = {"fifo": dq.SCHED_FIFO, "size": dq.SCHED_SIZE, "learned": dq.SCHED_LEARNED}
RMAT = {"even": (0.57, 0.19, 0.19), "skewed": (0.60, 0.15, 0.15)}  # quadrant probabilities a, b, c


# ------------------------------------------------------------------------------ the cases
def listed():
    return [
        # A small directed graph (a co-authorship or dependency graph of a thousand vertices)
        # searched from its file: latency of a whole call, most of it outside the kernels.
        {"name": "search_er1000", "kind": "search", "n": 1000, "degree": 10.0, "sets": 5, "low": 12, "high": 12,
         "density": 0.95, "gamma_out": 0.8, "gamma_in": 0.8, "min_size": 10},
        # The same size on an open handle: the smallest enumeration, bound by launches.
        {"name": "enum_er1000", "kind": "enum", "n": 1000, "degree": 10.0, "sets": 5, "low": 12, "high": 12,
         "density": 0.95, "gamma_out": 0.8, "gamma_in": 0.8, "min_size": 10, "schedule": "size"},
        # Many small graphs at once (neighbourhoods, communities): short tasks by the hundred
        # thousand, stack order, the batched form's plain schedule.
        {"name": "batch_fifo", "kind": "batch", "graphs": 64, "smallest": 200, "largest": 5000, "degree": 8.0,
         "low": 10, "high": 25, "density": 0.92, "gamma_out": 0.85, "gamma_in": 0.85, "min_size": 10,
         "schedule": "fifo", "resident_steps": 0},
        # A smaller batch with the learned schedule and device-resident steps.
        {"name": "batch_resident", "kind": "batch", "graphs": 24, "smallest": 200, "largest": 5000, "degree": 8.0,
         "low": 10, "high": 25, "density": 0.92, "gamma_out": 0.85, "gamma_in": 0.85, "min_size": 10,
         "schedule": "learned", "resident_steps": 16},
        # Level-0 branches of a graph of 2^16 vertices in the dense part of the loop.
        {"name": "window_rmat16", "kind": "window", "n": 1 << 16, "arcs": 1 << 20, "quadrants": "even", "sets": 50,
         "low": 15, "high": 30, "density": 0.95, "gamma_out": 0.9, "gamma_in": 0.9, "min_size": 12, "first": 0.5,
         "steps": 256},
        # Depth-1 tasks of a graph of 2^15 vertices expanded in one launch, one workgroup each.
        {"name": "tasks_rmat15", "kind": "tasks", "n": 1 << 15, "arcs": 1 << 19, "quadrants": "even", "sets": 50,
         "low": 15, "high": 30, "density": 0.95, "gamma_out": 0.9, "gamma_in": 0.9, "min_size": 12, "first": 0.6,
         "steps": 128},
        # Bounded units, smallest graph first: LDS bitmaps with many tasks of mixed sizes;
        # the plain schedule; then graphs whose bitmaps live in HBM, with unequal degree
        # bounds, and the largest with the learned schedule (long tasks split into pieces).
        {"name": "unit_rmat15_size", "kind": "unit", "n": 1 << 15, "arcs": 1 << 19, "quadrants": "even", "sets": 50,
         "low": 15, "high": 30, "density": 0.95, "gamma_out": 0.9, "gamma_in": 0.9, "min_size": 12, "first": 0.7,
         "steps": 64, "depth": 2, "schedule": "size"},
        {"name": "unit_rmat17_learned", "kind": "unit", "n": 1 << 17, "arcs": 1 << 21, "quadrants": "skewed",
         "sets": 100, "low": 20, "high": 40, "density": 0.97, "gamma_out": 0.9, "gamma_in": 0.95, "min_size": 18,
         "first": 0.5, "steps": 64, "depth": 2, "schedule": "learned"},
        {"name": "unit_rmat18_learned", "kind": "unit", "n": 1 << 18, "arcs": 1 << 22, "quadrants": "even",
         "sets": 125, "low": 20, "high": 40, "density": 0.95, "gamma_out": 0.9, "gamma_in": 0.9, "min_size": 18,
         "first": 0.6, "steps": 64, "depth": 2, "schedule": "learned"},
        # One task of a small graph in a loop that may not allocate.
        {"name": "serve_task", "kind": "serve", "n": 2000, "degree": 8.0, "sets": 8, "low": 16, "high": 25,
         "density": 0.92, "gamma_out": 0.85, "gamma_in": 0.85, "min_size": 10},
        # The cost model over the tasks of a few batches, and one pass of its training.
        {"name": "predict_256k", "kind": "predict", "samples": 1 << 18},
        {"name": "train_16k", "kind": "train", "samples": 1 << 14, "epochs": 1, "batch": 1024},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["search", "enum", "batch", "window", "tasks", "unit", "unit", "unit", "serve", "predict", "train"])
    gamma = rng.choice([0.8, 0.85, 0.9])
    if kind in ("search", "enum"):
        low = rng.randint(11, 14)
        case = {"kind": kind, "n": _log_int(rng, 300, 6000), "degree": round(rng.uniform(6.0, 12.0), 3),
                "sets": rng.randint(2, 9), "low": low, "high": low + rng.randint(0, 4), "density": 0.95,
                "gamma_out": gamma, "gamma_in": gamma, "min_size": 10}
        if kind == "enum":
            case["schedule"] = rng.choice(["fifo", "size"])
        return case
    if kind == "batch":
        schedule = rng.choice(["fifo", "size", "learned"])
        return {"kind": kind, "graphs": _log_int(rng, 3, 60), "smallest": 200, "largest": _log_int(rng, 1000, 5000),
                "degree": round(rng.uniform(6.0, 10.0), 3), "low": 10, "high": rng.randint(14, 25), "density": 0.92,
                "gamma_out": 0.85, "gamma_in": rng.choice([0.85, 0.9]), "min_size": rng.randint(9, 11),
                "schedule": schedule, "resident_steps": rng.choice([0, rng.randint(3, 20)])}
    if kind == "serve":
        return {"kind": kind, "n": _log_int(rng, 500, 5000), "degree": round(rng.uniform(6.0, 10.0), 3),
                "sets": rng.randint(3, 9), "low": 14, "high": rng.randint(16, 25), "density": 0.92,
                "gamma_out": 0.85, "gamma_in": 0.85, "min_size": 10}
    if kind == "predict":
        return {"kind": kind, "samples": _log_int(rng, 1, 1 << 20)}
    if kind == "train":
        return {"kind": kind, "samples": _log_int(rng, 500, 1 << 14), "epochs": 1,
                "batch": rng.choice([256, 1000, 1024, 2048])}
    n = _log_int(rng, 9000, 150000)  # spans both bitmap variants
    case = {"kind": kind, "n": n, "arcs": int(n * rng.uniform(12.0, 16.0)), "quadrants": rng.choice(sorted(RMAT)),
            "sets": max(3, n // 1300), "low": 18, "high": rng.randint(24, 40), "density": 0.95,
            "gamma_out": 0.9, "gamma_in": rng.choice([0.9, 0.95]), "min_size": rng.randint(14, 18),
            "first": round(rng.uniform(0.3, 0.7), 3)}
    if kind == "window":
        case["steps"] = rng.randint(40, 256)
    elif kind == "tasks":
        case["steps"] = rng.randint(10, 100)
    else:
        case.update(steps=rng.randint(12, 64), depth=rng.choice([1, 2]), schedule=rng.choice(["fifo", "size", "learned"]))
    return case


# ----------------------------------------------------------------------------- the graphs
def _plant(rng, n, sets, low, high, density):
    """Arc keys (u * n + v) of `sets` disjoint planted quasi-cliques."""
    members, at, keys = rng.permutation(n), 0, []
    for _ in range(sets):
        size = int(rng.integers(low, high + 1))
        part = members[at:at + size].astype(np.int64)
        at += size
        hit = rng.random((len(part), len(part))) < density
        np.fill_diagonal(hit, False)
        u, v = np.nonzero(hit)
        keys.append(part[u] * n + part[v])
    return np.concatenate(keys) if keys else np.zeros(0, np.int64)


def _er_arcs(rng, n, degree):
    count = rng.binomial(n * (n - 1), min(1.0, degree / (n - 1)))
    u, v = rng.integers(0, n, count), rng.integers(0, n, count)
    return (u * n + v)[u != v]


def _rmat_arcs(seed, n, arcs, quadrants):
    """`arcs` distinct R-MAT arc keys on n vertices (ids at or above n are drawn again)."""
    a, b, c = RMAT[quadrants]
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    keys = torch.zeros(0, dtype=torch.int64, device=DEVICE)
    while keys.numel() < arcs:
        m = int((arcs - keys.numel()) * 1.3) + 1024
        u = torch.zeros(m, dtype=torch.int64, device=DEVICE)
        v = torch.zeros(m, dtype=torch.int64, device=DEVICE)
        for _ in range((n - 1).bit_length()):
            x = torch.rand(m, generator=g, device=DEVICE, dtype=torch.float64)
            u = 2 * u + (x >= a + b)
            v = 2 * v + (((x >= a) & (x < a + b)) | (x >= a + b + c))
        fresh = (u * n + v)[(u != v) & (u < n) & (v < n)]
        keys = torch.unique(torch.cat([keys, fresh]))
        if keys.numel() > arcs:
            keys = keys[torch.randperm(keys.numel(), generator=g, device=DEVICE)[:arcs]]
    return keys.cpu().numpy()


def _graph(case, seed):
    """Vertex count and the sorted distinct arc keys of the case's graph."""
    rng, n = np.random.default_rng(seed), case["n"]
    if "arcs" in case:
        keys = _rmat_arcs(seed, n, case["arcs"], case["quadrants"])
    else:
        keys = _er_arcs(rng, n, case["degree"])
    planted = _plant(rng, n, case["sets"], case["low"], case["high"], case["density"])
    return n, np.unique(np.concatenate([keys, planted]))


def _csr(n, keys):
    """Out- and in-lists as (offsets, ids) pairs."""
    u, v = np.divmod(keys, n)
    back = np.sort(v * n + u)
    out = []
    for k in (keys, back):
        src, dst = np.divmod(k, n)
        off = np.zeros(n + 1, np.uint64)
        off[1:] = np.cumsum(np.bincount(src, minlength=n))
        out.append((off, dst.astype(np.int32)))
    return out


def _write_text(path, n, keys):
    u, v = np.divmod(keys, n)
    at = np.searchsorted(u, np.arange(n + 1))
    ids = [str(x) for x in v.tolist()]
    with open(path, "w") as f:
        f.write("".join(" ".join(ids[at[i]:at[i + 1]]) + "\n" for i in range(n)))


# ------------------------------------------------------------------- handles and their data
class Handle(dq.Engine):
    """An open handle that is closed with the program's last reference to it."""

    def __del__(self):
        self.close()


def _i32(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_int32))


def _u32(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32))


def _u64(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_uint64))


def _open(schedule="size", resident_steps=0):
    cfg = dq.Config()
    cfg.host_addfail_check = 1
    cfg.schedule = SCHEDULES[schedule]
    cfg.resident_steps = resident_steps
    eng = Handle(cfg)
    if schedule == "learned":
        eng.set_cost_model(learn.load_model())
    return eng


def _prepare_graph(eng, n, keys, case):
    (oo, on), (io, inb) = _csr(n, keys)
    k = ctypes.c_int32()
    eng._check(eng.lib.dqc_prepare_graph(eng.h, n, _u64(oo), _i32(on), _u64(io), _i32(inb), None, None, None, None, 0,
                                         case["gamma_out"], case["gamma_in"], case["min_size"], ctypes.byref(k), None),
               "dqc_prepare_graph")
    return k.value


def _stack(eng):
    """The task stack: meta (tasks x 9) and records (x 6) as arrays."""
    nt, nr = ctypes.c_int64(), ctypes.c_int64()
    eng._check(eng.lib.dqc_fetch_tasks(eng.h, ctypes.byref(nt), ctypes.byref(nr), None, None), "dqc_fetch_tasks")
    meta, rec = np.zeros((nt.value, 9), np.int32), np.zeros((nr.value, 6), np.uint32)
    if nt.value:
        eng._check(eng.lib.dqc_fetch_tasks(eng.h, ctypes.byref(nt), ctypes.byref(nr), _i32(meta), _u32(rec)),
                   "dqc_fetch_tasks")
    return meta, rec


def _cliques(eng):
    """Raw cliques as (sizes, ids)."""
    count, total = ctypes.c_int64(), ctypes.c_int64()
    eng._check(eng.lib.dqc_fetch_cliques(eng.h, ctypes.byref(count), ctypes.byref(total), None, None),
               "dqc_fetch_cliques")
    sizes, ids = np.zeros(count.value, np.int32), np.zeros(total.value, np.int32)
    if count.value:
        eng._check(eng.lib.dqc_fetch_cliques(eng.h, ctypes.byref(count), ctypes.byref(total), _i32(sizes), _i32(ids)),
                   "dqc_fetch_cliques")
    return sizes, ids


def _mixed(words):
    """A 64-bit mix of each word, for ordering pieces of data by content."""
    x = words.astype(np.uint64) * np.uint64(0x9E3779B97F4A7C15)
    x ^= x >> np.uint64(29)
    x *= np.uint64(0xBF58476D1CE4E5B9)
    return x ^ (x >> np.uint64(32))


def _sorted_sets(sizes, ids):
    """The sets with ascending ids, shorter sets first, in one order for the same sets."""
    if not len(sizes):
        return sizes, ids
    lengths = sizes.astype(np.int64)
    ids = ids[np.lexsort((ids, np.repeat(np.arange(len(lengths)), lengths)))]
    starts = np.cumsum(lengths) - lengths
    order = np.lexsort((np.add.reduceat(_mixed(ids), starts), lengths))
    return sizes[order], np.concatenate([ids[i:i + l] for i, l in zip(starts[order], lengths[order])])


def _sorted_tasks(meta, rec):
    """The tasks' (size, members, mode) rows and their records, in one order for the same
    tasks: by member count, then by the member ids (no two tasks have the same members)."""
    if not len(meta):
        return meta[:, 1:4], rec
    starts, sizes, members = (meta[:, i].astype(np.int64) for i in range(3))
    before = np.cumsum(members) - members
    ids = rec[np.repeat(starts - before, members) + np.arange(int(members.sum())), 0]
    order = np.lexsort((np.add.reduceat(_mixed(ids), before), members))
    return meta[order, 1:4], np.concatenate([rec[i:i + l] for i, l in zip(starts[order], sizes[order])])


# Room a program keeps for results: (sets, their ids, tasks, their records, bytes of maximal files)
ROOM = {"sets": 1 << 15, "ids": 1 << 19, "tasks": 1 << 17, "records": 1 << 21, "bytes": 1 << 23}


def _keep(state, name, data):
    """`data` in the state's buffer of that name, which holds zeros beyond it."""
    buf, count = state["room"].get(name), len(data)
    size = ROOM[name]
    while size < count:
        size *= 2
    if buf is None or len(buf) < size:
        buf = state["room"][name] = np.zeros((size,) + data.shape[1:], data.dtype)
    used = state["used"].get(name, 0)
    buf[:count] = data
    if used > count:
        buf[count:used] = 0
    state["used"][name] = count
    return buf


def _push(eng, rec, members, mode, covered=0):
    """dqc_push_root for a level-0 task, dqc_push_task for the others."""
    if mode == 0:
        eng._check(eng.lib.dqc_push_root(eng.h, _u32(rec), len(rec), covered), "dqc_push_root")
    else:
        eng._check(eng.lib.dqc_push_task(eng.h, _u32(rec), len(rec), members, covered, mode), "dqc_push_task")


# -------------------------------------------------------------- the allocation-free entry
class TaskDesc(ctypes.Structure):
    """dqc_task_desc of include/dqc.h."""
    _fields_ = [("offset", ctypes.c_uint64), ("size", ctypes.c_int32), ("members", ctypes.c_int32),
                ("covered", ctypes.c_int32), ("mode", ctypes.c_int32), ("steps", ctypes.c_int32),
                ("flags", ctypes.c_int32), ("id", ctypes.c_uint32), ("parent", ctypes.c_uint32),
                ("depth", ctypes.c_uint16), ("graph", ctypes.c_uint16), ("dmin_out", ctypes.c_uint16),
                ("dmax_out", ctypes.c_uint16), ("dmin_in", ctypes.c_uint16), ("dmax_in", ctypes.c_uint16),
                ("first_step", ctypes.c_int32)]


class DeviceGraph(ctypes.Structure):
    """dqc_device_graph of include/dqc.h."""
    _fields_ = [("n", ctypes.c_int32), ("out_off", ctypes.c_void_p), ("out_nbr", ctypes.c_void_p),
                ("in_off", ctypes.c_void_p), ("in_nbr", ctypes.c_void_p), ("two_off", ctypes.c_void_p),
                ("two_nbr", ctypes.c_void_p), ("md_out", ctypes.c_void_p), ("md_in", ctypes.c_void_p),
                ("ub_out", ctypes.c_void_p), ("ub_in", ctypes.c_void_p), ("table_len", ctypes.c_int32),
                ("min_size", ctypes.c_int32), ("host_addfail_check", ctypes.c_int32)]


SERVE_TASKS, SERVE_RECORDS, SERVE_SETS, SERVE_IDS = 1 << 12, 1 << 18, 1 << 12, 1 << 15


def _device(array):
    return torch.from_numpy(np.ascontiguousarray(array)).to(DEVICE)


def _prepare_serve(case, seed):
    """A condensed graph, its tables and its costliest level-1 task in device memory, and
    room for the results."""
    n, keys = _graph(case, seed)
    go, gi, mn = case["gamma_out"], case["gamma_in"], case["min_size"]
    with tempfile.TemporaryDirectory() as folder:
        path = os.path.join(folder, "graph.txt")
        _write_text(path, n, keys)
        lists = dq.load_graph(path)
        _, _, orig = dq.level0(path, go, gi, mn)
    rank = {v: i for i, v in enumerate(orig)}
    k = len(orig)
    graph, keep = DeviceGraph(), []
    graph.n = k
    for name in ("out", "in", "two"):
        rows = [sorted(rank[x] for x in lists[name][v] if x in rank) for v in orig]
        off = np.zeros(k + 1, np.int64)
        off[1:] = np.cumsum([len(r) for r in rows])
        nbr = np.array([x for r in rows for x in r] + [0], np.int32)
        for key, data in ((name + "_off", off), (name + "_nbr", nbr)):
            keep.append(_device(data))
            setattr(graph, key, keep[-1].data_ptr())
    length = 2 * (max(k, mn) + 2) + 2
    tables = {"md_out": dq.min_degrees(go, length - 1), "md_in": dq.min_degrees(gi, length - 1),
              "ub_out": [int(d / go) for d in range(length)], "ub_in": [int(d / gi) for d in range(length)]}
    for key, data in tables.items():
        keep.append(_device(np.array(data, np.int32)))
        setattr(graph, key, keep[-1].data_ptr())
    graph.table_len, graph.min_size, graph.host_addfail_check = length, mn, 1
    with _open() as eng:
        _prepare_graph(eng, n, keys, case)
        eng.step(1)
        meta, rec = _stack(eng)
    rows, rec = _sorted_tasks(meta, rec)
    pick = int(np.argmax(rows[:, 0]))
    size, members, mode = (int(x) for x in rows[pick])
    end = int(rows[:pick + 1, 0].sum())
    desc = TaskDesc(0, size, members, 0, mode, size - members, 0, 0, 0xFFFFFFFF, 1, 0, 0, 0, 0, 0, 0)
    state = {"graph": graph, "keep": keep, "size": size, "desc": _device(np.frombuffer(bytes(desc), np.int32).copy()),
             "rec": _device(rec[end - size:end].view(np.int32)),
             "tasks": torch.zeros((SERVE_TASKS, 14), dtype=torch.int32, device=DEVICE),
             "records": torch.zeros((SERVE_RECORDS, 6), dtype=torch.int32, device=DEVICE),
             "ids": torch.zeros(SERVE_IDS, dtype=torch.int32, device=DEVICE),
             "sets": torch.zeros(SERVE_SETS, dtype=torch.int64, device=DEVICE),
             "counters": torch.zeros(9, dtype=torch.int64, device=DEVICE), "call": dq.load().dqc_expand_noalloc}
    i64, ptr = ctypes.c_int64, ctypes.c_void_p
    state["call"].restype = ctypes.c_int32
    state["call"].argtypes = [ctypes.POINTER(DeviceGraph), ptr, ptr, i64, i64, ctypes.c_int32, ptr, ptr, i64, i64, ptr,
                              ptr, i64, i64, ptr, ptr]
    return state


def _run_serve(s):
    rc = s["call"](ctypes.byref(s["graph"]), s["desc"].data_ptr(), s["rec"].data_ptr(), 1, s["size"], s["size"],
                   s["tasks"].data_ptr(), s["records"].data_ptr(), SERVE_TASKS, SERVE_RECORDS, s["ids"].data_ptr(),
                   s["sets"].data_ptr(), SERVE_SETS, SERVE_IDS, s["counters"].data_ptr(),
                   torch.cuda.current_stream().cuda_stream)
    if rc != dq.DQC_OK:
        raise dq.DQCError(f"dqc_expand_noalloc failed: {rc}")
    # one task's children and cliques come in the order of its branches; a clique is a set:
    # its ids are put in ascending order (the cliques lie end to end)
    ends = (s["sets"] >> 24) + (s["sets"] & 0xFFFFFF)
    owner = torch.zeros(SERVE_IDS + 1, dtype=torch.int64, device=DEVICE)
    owner.index_add_(0, ends.clamp(max=SERVE_IDS), torch.ones_like(ends))
    key = (torch.cumsum(owner[:-1], 0) << 32) + s["ids"]
    return {"tasks": s["tasks"], "records": s["records"], "sets": s["sets"], "ids": torch.sort(key).values & 0xFFFFFFFF,
            "counters": s["counters"]}


# --------------------------------------------------------------------------- cost model
def _task_shapes(rng, n):
    """Features of n tasks as a task log gives them, and log1p of the branches each ran."""
    members = 1 + rng.geometric(0.25, n)
    size = members + np.exp(rng.uniform(np.log(2.0), np.log(9000.0), n)).astype(np.int64)
    depth = np.minimum(members, 1 + rng.geometric(0.5, n))
    low_out, low_in = (rng.integers(9, 18, n) for _ in range(2))
    high_out, high_in = (np.minimum(size, low_out + (size * rng.uniform(0.05, 0.9, n)).astype(np.int64))
                         for _ in range(2))
    x = np.log1p(np.stack([members, size - members, depth, low_out, high_out, low_in, high_in], 1)).astype(np.float32)
    branches = ((size - members) * rng.uniform(0.3, 1.0, n)).astype(np.int64)
    return x, np.log1p(branches).astype(np.float32)


def _shuffled(n, epochs, seed):
    """The sample order of each epoch: a Fisher-Yates shuffle driven by std::mt19937_64."""
    mask, state = (1 << 64) - 1, [seed & ((1 << 64) - 1)]
    for i in range(1, 312):
        state.append((6364136223846793005 * (state[-1] ^ (state[-1] >> 62)) + i) & mask)
    at, order, orders = 312, list(range(n)), []
    for _ in range(epochs):
        for i in range(n - 1, 0, -1):
            if at == 312:
                for j in range(312):
                    y = (state[j] & 0xFFFFFFFF80000000) | (state[(j + 1) % 312] & 0x7FFFFFFF)
                    state[j] = state[(j + 156) % 312] ^ (y >> 1) ^ (0xB5026F5AA96619E9 if y & 1 else 0)
                at = 0
            y = state[at]
            at += 1
            y ^= (y >> 29) & 0x5555555555555555
            y ^= (y << 17) & 0x71D67FFFEDA60000
            y ^= (y << 37) & 0xFFF7EEE000000000
            y ^= y >> 43
            r = y % (i + 1)
            order[i], order[r] = order[r], order[i]
        orders.append(np.array(order))
    return orders


def _layers(p):
    h, i = dq.MLP_HIDDEN, dq.MLP_IN
    cut = np.cumsum([h * i, h, h * h, h, h])
    w1, b1, w2, b2, w3, b3 = np.split(p, cut)
    return w1.reshape(h, i), b1, w2.reshape(h, h), b2, w3, b3


def _forward64(p, x):
    w1, b1, w2, b2, w3, b3 = _layers(p)
    a = np.maximum(x @ w1.T + b1, 0.0)
    b = np.maximum(a @ w2.T + b2, 0.0)
    return a, b, b @ w3 + b3[0]


def _train64(p, x, t, epochs, batch, lr, seed):
    """Adam on minibatches, in float64: (parameters, final mean squared error)."""
    p, m, v, step = p.copy(), np.zeros_like(p), np.zeros_like(p), 0
    lr, b1, b2 = float(np.float32(lr)), float(np.float32(0.9)), float(np.float32(0.999))
    for order in _shuffled(len(x), epochs, seed):
        for s in range(0, len(x), batch):
            xs, ts = x[order[s:s + batch]], t[order[s:s + batch]]
            _, _, w2, _, w3, _ = _layers(p)
            a, b, y = _forward64(p, xs)
            dy = 2.0 * (y - ts) / len(xs)
            db = np.where(b > 0, dy[:, None] * w3, 0.0)
            da = np.where(a > 0, db @ w2, 0.0)
            g = np.concatenate([(da.T @ xs).ravel(), da.sum(0), (db.T @ a).ravel(), db.sum(0), dy @ b, [dy.sum()]])
            step += 1
            m, v = b1 * m + (1 - b1) * g, b2 * v + (1 - b2) * g * g
            p -= lr * (m / (1 - b1 ** step)) / (np.sqrt(v / (1 - b2 ** step)) + 1e-8)
    return p, float(np.mean((_forward64(p, x)[2] - t) ** 2))


LEARNING_RATE = 2e-3


# ------------------------------------------------------------------------------- one case
def _prepare_search(case, seed):
    n, keys = _graph(case, seed)
    folder = tempfile.TemporaryDirectory()
    path = os.path.join(folder.name, "graph.txt")
    _write_text(path, n, keys)
    return {"folder": folder, "path": path, "result": os.path.join(folder.name, "maximal.txt")}


def _prepare_batch(case, seed):
    rng = np.random.default_rng(seed)
    eng = _open(case["schedule"], case["resident_steps"])
    low, high = math.log(case["smallest"]), math.log(case["largest"])
    folder = tempfile.TemporaryDirectory()
    paths = []
    for g in range(case["graphs"]):
        n = int(round(math.exp(rng.uniform(low, high))))
        sets = 1 + int(rng.integers(0, 10))
        keys = np.concatenate([_er_arcs(rng, n, case["degree"]),
                               _plant(rng, n, sets, case["low"], case["high"], case["density"])])
        paths.append(os.path.join(folder.name, f"graph{g}.txt"))
        _write_text(paths[-1], n, np.unique(keys))
    sizes = eng.prepare_batch(paths, case["gamma_out"], case["gamma_in"], case["min_size"])
    # the level-0 task of every graph that keeps any vertex, with the graph's own ids
    meta, rec = _stack(eng)
    roots, base, tasks = [], 0, iter(meta)
    for g, size in enumerate(sizes):
        if size:
            at = next(tasks)
            own = rec[at[0]:at[0] + at[1]].copy()
            own[:, 0] -= np.uint32(base)
            roots.append((g, own, int(at[8])))
        base += (size + 31) // 32 * 32
    return {"eng": eng, "folder": folder, "roots": roots,
            "results": [os.path.join(folder.name, f"maximal{g}.txt") for g in range(len(paths))]}


def _prepare_handle(case, seed):
    """An open handle with the graph, and what run() queues: the level-0 task, or (kind
    "tasks") the depth-1 tasks of the window."""
    n, keys = _graph(case, seed)
    eng = _open(case.get("schedule", "fifo"))
    k = _prepare_graph(eng, n, keys, case)
    meta, rec = _stack(eng)
    work = [(rec, 0, 0, int(meta[0][8]))] if len(meta) else []
    if "first" in case and work:
        eng.set_unit(int(case["first"] * k), case["steps"], case.get("depth", 0))
    if case["kind"] == "tasks" and work:
        eng.step(1)
        rows, rec = _sorted_tasks(*_stack(eng))
        ends = np.cumsum(rows[:, 0])
        work = [(rec[e - s:e].copy(), int(nm), int(mode), 0) for e, (s, nm, mode) in zip(ends, rows)]
    return {"eng": eng, "work": work}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "search":
        state = _prepare_search(case, seed)
    elif kind == "batch":
        state = _prepare_batch(case, seed)
    elif kind == "serve":
        state = _prepare_serve(case, seed)
    elif kind == "predict":
        x, _ = _task_shapes(np.random.default_rng(seed), case["samples"])
        state = {"params": learn.load_model(), "x": x}
    elif kind == "train":
        x, t = _task_shapes(np.random.default_rng(seed), case["samples"])
        state = {"params": dq.mlp_init(seed), "x": x, "t": t, "seed": seed}
    else:
        state = _prepare_handle(case, seed)
    state.update(case=case, room={}, used={})
    return state


def _result_bytes(path):
    return np.fromfile(path, np.uint8) if os.path.exists(path) else np.zeros(0, np.uint8)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "search":
        count, st = dq.search_file(state["path"], case["gamma_out"], case["gamma_in"], case["min_size"], None,
                                   state["result"])
        return {"count": count, "tasks": st.tasks_expanded, "branches": st.branches,
                "maximal": _keep(state, "bytes", _result_bytes(state["result"]))}
    if kind == "serve":
        return _run_serve(state)
    if kind == "predict":
        return dq.mlp_forward(state["params"], state["x"])
    if kind == "train":
        params, loss = dq.mlp_train(state["params"], state["x"], state["t"], epochs=case["epochs"], batch=case["batch"],
                                    lr=LEARNING_RATE, seed=state["seed"])
        return {"params": params, "loss": loss}
    eng = state["eng"]
    eng.reset()
    if kind == "batch":
        for g, rec, covered in state["roots"]:
            eng._check(eng.lib.dqc_push_graph_root(eng.h, g, _u32(rec), len(rec), covered), "dqc_push_graph_root")
        eng.run(SCHEDULES[case["schedule"]])
        counts, st = eng.finish_batch(state["results"])
        return {"counts": np.array(counts), "tasks": st.tasks_expanded, "branches": st.branches, "raw": st.raw_cliques,
                "maximal": _keep(state, "bytes", np.concatenate([_result_bytes(p) for p in state["results"]]))}
    for rec, members, mode, covered in state["work"]:
        _push(eng, rec, members, mode, covered)
    if kind in ("window", "tasks"):
        if state["work"]:
            eng.step(1, SCHEDULES["fifo"])
    else:
        eng.run(SCHEDULES[case["schedule"]])
    st = eng.stats()
    sizes, ids = _sorted_sets(*_cliques(eng))
    out = {"expanded": st.tasks_expanded, "branches": st.branches, "raw": st.raw_cliques,
           "truncated": st.truncated_children, "sizes": _keep(state, "sets", sizes), "ids": _keep(state, "ids", ids)}
    if kind in ("window", "tasks"):
        children, records = _sorted_tasks(*_stack(eng))
        out.update(children=_keep(state, "tasks", children), records=_keep(state, "records", records))
    return out


def work(case):
    """Bytes and operations of one pass that no enumeration of the case can do without: the
    graph's lists and the level-0 task read once (the enumeration's own work depends on the
    graph, not on its sizes alone); for the model, its samples, parameters and products."""
    kind = case["kind"]
    if kind in ("predict", "train"):
        rows = case["samples"] * case.get("epochs", 1)
        layers = dq.MLP_IN * dq.MLP_HIDDEN + dq.MLP_HIDDEN * dq.MLP_HIDDEN + dq.MLP_HIDDEN
        if kind == "predict":
            return {"bytes": 4 * rows * (dq.MLP_IN + 1) + 4 * dq.MLP_PARAMS, "flops": 2 * rows * layers}
        return {"bytes": 4 * rows * (dq.MLP_IN + 1) + 8 * dq.MLP_PARAMS, "flops": 6 * rows * layers}
    if kind == "batch":  # the mean of a log-uniform size
        low, high = case["smallest"], case["largest"]
        n = case["graphs"] * (high - low) / math.log(max(high, low + 1) / low)
        arcs = n * case["degree"]
    elif "arcs" in case:
        n, arcs = case["n"], case["arcs"]
    else:
        n, arcs = case["n"], case["n"] * case["degree"]
    return {"bytes": 2 * 4 * arcs + 3 * 8 * n + 24 * n, "flops": 0}


def exact(case, seed):
    kind = case["kind"]
    if kind == "predict":
        x, _ = _task_shapes(np.random.default_rng(seed), case["samples"])
        return _forward64(learn.load_model().astype(np.float64), x.astype(np.float64))[2]
    if kind == "train":
        x, t = _task_shapes(np.random.default_rng(seed), case["samples"])
        params, loss = _train64(dq.mlp_init(seed).astype(np.float64), x.astype(np.float64), t.astype(np.float64),
                                case["epochs"], case["batch"], LEARNING_RATE, seed)
        return {"params": params, "loss": loss}
    return None  # sets, task records and counts: whole numbers
