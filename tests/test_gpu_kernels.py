"""Edge sizes of single kernels and dispatch rules, against the CPU oracle (bit-exact for
BFS, SSSP and CC)."""
import numpy as np
import pytest

from conftest import random_graph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 31, 255, 257, 65537, 262145, 524321])
def test_frontier_slices_cover_ragged_graphs(mg, oracle, device, n):
    # vertex counts around one slice, one workgroup and the 1024-workgroup share
    g = random_graph(mg, n, 6 * n, seed=n, symmetric=n % 2 == 1, wmax=16)
    src = int(np.argmax(g.degrees()))
    srcs = [src, n - 1, 0]
    with mg.Graph(g, symmetric=n % 2 == 1) as dg:
        assert np.array_equal(dg.bfs(src), oracle.bfs(g.row_offsets, g.col_idx, src))
        assert np.array_equal(dg.sssp(src), oracle.sssp(g.row_offsets, g.col_idx, g.values, src))
        for got, s in zip(dg.bfs_batch(srcs), srcs):
            assert np.array_equal(got, oracle.bfs(g.row_offsets, g.col_idx, s))
        for got, s in zip(dg.sssp_batch(srcs), srcs):
            assert np.array_equal(got, oracle.sssp(g.row_offsets, g.col_idx, g.values, s))
