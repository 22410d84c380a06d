"""Device buffers kept between handles: searches one after another and in several threads at
once, on graphs of different sizes, give the results of the first search; so do cost-model calls
between them."""
import os
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from tests.conftest import GOLDEN

pytestmark = pytest.mark.gpu

NAMES = ["workload1", "workload3_g0", "rand088", "bigk20000"]


def search(dqc, manifest, tmp_path, name, tag):
    c = next(x for x in manifest["cases"] if x["name"] == name)
    out = str(tmp_path / f"{name}_{tag}.max")
    cnt, st = dqc.search_file(os.path.join(GOLDEN, c["graph"]), c["out_gamma"], c["in_gamma"], c["min_size"], None, out)
    got = open(out, "rb").read() if os.path.exists(out) else b""
    want = open(os.path.join(GOLDEN, c["expected"]), "rb").read() if c["expected"] else b""
    return got == want and cnt == c["maximal"] and st.tasks_expanded == c["tasks"]


def test_buffers_pass_between_handles(dqc, manifest, tmp_path):
    for i in range(3):
        for name in NAMES:
            assert search(dqc, manifest, tmp_path, name, i), (name, i)


def test_buffers_pass_between_threads(dqc, manifest, tmp_path):
    p, x = dqc.mlp_init(1), np.random.default_rng(0).uniform(0, 5, (5000, 7)).astype(np.float32)
    y = dqc.mlp_forward(p, x)
    with ThreadPoolExecutor(4) as pool:
        runs = [pool.submit(search, dqc, manifest, tmp_path, NAMES[i % 4], f"t{i}") for i in range(16)]
        model = [pool.submit(dqc.mlp_forward, p, x) for _ in range(8)]
        assert all(r.result() for r in runs)
        assert all(np.array_equal(m.result(), y) for m in model)
