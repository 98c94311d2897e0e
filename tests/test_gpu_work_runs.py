"""GPU: the batched path's persistent kernels hand every task to one wave.

Grids below, at and above the work queue's eight counters (a block is four
waves), so that counters start with unequal numbers of waves, some with none,
and runs of one and of many tasks occur; level rows and counts against the
oracle's vertex-level walk."""
import numpy as np
import pytest

import oracle
from gem_amd import GemContext, Graph, Query

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def case():
    g = Graph.rmat(13, 12.0, 5, 4111)
    qs, i = [], 0
    while len(qs) < 5:
        q = Query.random_walk(g, 3 + len(qs) % 3, 900 + i)
        i += 1
        if q.num_e >= 2:
            qs.append(q)
    refs = []
    for q in qs:
        r = oracle.count(g, q)
        refs.append(oracle.vcount(g, q, oracle.vertex_order_from_edges(q, r["order"])))
    return g, qs, refs


@pytest.mark.parametrize("blocks,heavy,graph", [(1, None, False), (2, (32, 64), False), (3, (32, 64), True),
                                                (17, None, True), (2048, (32, 64), False)])
def test_every_task_runs_once(case, blocks, heavy, graph):
    g, qs, refs = case
    with GemContext(0) as ctx:
        ctx.load_data(g)
        ctx.set_persistent_blocks(blocks)
        ctx.set_graph(graph)
        if heavy:
            ctx.set_heavy_split(*heavy)
        for _ in range(2):
            for q, r, ref in zip(qs, ctx.match_batch(qs), refs):
                assert r["count"] == ref["count"]
                assert np.array_equal(r["level_rows"], ref["level_rows"])
