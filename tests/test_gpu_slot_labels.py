"""GPU: byte labels with and without the labels of the adjacency slots (the
array's limit on either side of its size), neighbours in HBM and in host memory:
the array takes device memory only when it is made, and candidates, tables and
counts equal the oracle's either way."""
import numpy as np
import pytest

import oracle
from gem_amd import GemContext
from test_gpu_filter_edges import _graph, _queries

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def case():
    """The graph of the filter's edge cases, and per query its candidates at
    threshold 0 and 1, table sizes and tables."""
    g = _graph(3)
    ref = []
    for q in _queries(3):
        lists = [oracle.filter(g, q, threshold=t) for t in (0, 1)]
        sizes = oracle.table_sizes(g, q)
        tables = [oracle.edge_table(g, q, d, len(lists[0][int(q.edges[d // 2][d % 2])]), int(sizes[d]))
                  for d in range(2 * q.num_e)]
        ref.append((q, lists, sizes, tables))
    return g, ref


def _loaded(g, host, limit):
    """A context with the graph, and the device memory that its load took."""
    ctx = GemContext(0)
    ctx.set_graph_residency(host)
    ctx.set_slot_labels(limit)
    before = ctx.memory_stats()["in_use"]
    ctx.load_data(g)
    return ctx, ctx.memory_stats()["in_use"] - before


@pytest.mark.parametrize("host", [False, True])
@pytest.mark.parametrize("over", [None, 16, 15, 0])  # limit: none, the array's size, one below, leave it out
def test_with_and_without(case, host, over):
    g, ref = case
    ctx0, bytes0 = _loaded(g, host, 0)
    ctx0.close()
    if host:  # offsets, labels and the ids of at most all vertices (and the allocator's rounding)
        assert bytes0 < 13 * g.num_vertices + 3 * (1 << 16)
    ctx, took = _loaded(g, host, None if over is None else 0 if over == 0 else g.num_slots + over)
    with ctx:
        if over in (None, 16):
            # (size classes a quarter apart below 1 MiB, 64 KiB units above)
            assert g.num_slots <= took - bytes0 <= 1.25 * g.num_slots + (1 << 16)
        else:
            assert took == bytes0
        for q, lists, sizes, tables in ref:
            for t in (1, 0):
                _, got = ctx.filter(q, threshold=t)
                for u in range(q.num_v):
                    assert np.array_equal(got[u], lists[t][u])
            num = [len(x) for x in lists[0]]
            assert np.array_equal(ctx.build_edge_tables(), sizes)
            for d, table in enumerate(tables):
                if table is None:  # keyed on a leaf
                    continue
                off, val = ctx.read_edge_table(d, num[int(q.edges[d // 2][d % 2])], int(sizes[d]))
                assert np.array_equal(off, table[0]) and np.array_equal(val, table[2])
