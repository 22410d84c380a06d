"""The device pass before the maximal-set filter: the maximal file of a search that keeps no raw
file (raw cliques filtered on the device first, from 4,096 of them on) equals the one of a search
that writes them all (host filter alone), and the host filter's result on that raw file."""
import os

import pytest

from tests.test_gpu_rows import CASES, cluster_graph, write

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", [5, 7, 8, 9])  # 2,320 raw cliques (host filter alone), 42,357, 42,689, 6,168
def test_maximal_file_with_and_without_raw_file(dqc, tmp_path, case):
    sizes, density, links, go, gi, mn = CASES[case]
    path = str(tmp_path / "g.txt")
    write(path, cluster_graph(100 + case, sizes, density, links))
    files = {k: str(tmp_path / k) for k in ("raw", "with_raw", "without", "again", "batch")}
    count, st = dqc.search_file(path, go, gi, mn, files["raw"], files["with_raw"])
    count2, st2 = dqc.search_file(path, go, gi, mn, None, files["without"])
    counts, _ = dqc.search_batch([path, path], go, gi, mn, [files["batch"], None])
    assert count == count2 and counts == [count, count] and st.raw_cliques == st2.raw_cliques
    assert dqc.remove_non_max(files["raw"], files["again"]) == count
    want = open(files["again"], "rb").read()
    for k in ("with_raw", "without", "batch"):
        assert open(files[k], "rb").read() == want, k
    assert os.path.getsize(files["raw"]) > 0
