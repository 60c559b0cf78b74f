"""Results reach the caller's memory whole, whatever their size: one piece of
32 KiB and its neighbours, the halves of the pinned ring (4 MiB each) and more
than both, arrays that do not start on 16 bytes, and calls on several threads."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PIECE, HALF = (32 << 10) // 4, (4 << 20) // 4


def sparse_graph(gsw, n):
    src = np.arange(0, n - 1, 3, dtype=np.int32)
    return gsw.from_edges(n, src, src + 1)


@pytest.mark.parametrize("n", [2, 5, PIECE - 1, PIECE, PIECE + 1, 3 * PIECE + 7, HALF - 1, HALF,
                               HALF + 1, 2 * HALF, 2 * HALF + 3, 5 * HALF + 11])
def test_labels_of_every_size(gsw, n):
    h = sparse_graph(gsw, n)
    g = gsw.Graph(h)
    want = np.arange(n, dtype=np.int32)
    want[np.arange(0, n - 1, 3) + 1] -= 1
    for _ in range(2):
        assert np.array_equal(g.cc(), want)
    g.close()


@pytest.mark.parametrize("n", [7, 4097, 300001])
def test_several_arrays_unaligned(gsw, orc, n):
    h = sparse_graph(gsw, n)
    g = gsw.Graph(h)
    lv, nsp, dep = g.bc(0)
    ref = orc.bfs(h.row_ptr, h.col, 0)
    assert np.array_equal(lv, ref)
    assert np.array_equal(nsp, (ref >= 0).astype(float))
    want = np.zeros(n)
    want[0] = 1.0
    assert np.array_equal(dep, want)
    off = np.array([0, n // 3 * 3, n] if n % 3 else [0, n], np.int64)
    lv, lab = g.batch_bfs_cc(off)
    assert lv[0] == 0 and lv[1] == 1 and lab[1] == 0 and lab[2] == 2
    g.close()


def test_threads_share_the_rings(gsw):
    sizes = [HALF + 5, 3 * HALF, 100, 2 * PIECE + 1]
    graphs = [(n, gsw.Graph(sparse_graph(gsw, n))) for n in sizes]
    bad = []

    def work(n, g):
        want = np.arange(n, dtype=np.int32)
        want[np.arange(0, n - 1, 3) + 1] -= 1
        for _ in range(6):
            if not np.array_equal(g.cc(), want):
                bad.append(n)

    th = [threading.Thread(target=work, args=a) for a in graphs]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad
    for _, g in graphs:
        g.close()
    # every handle gone: the rings went with them, and come back
    n = 2 * HALF
    g = gsw.Graph(sparse_graph(gsw, n))
    assert g.cc()[1] == 0
    g.close()
