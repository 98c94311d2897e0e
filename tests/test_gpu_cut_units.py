"""GPU: write walks whose 64-row units cost more than a run are cut between rows.

A dense graph of few labels, so that lists are long (units of up to tens of
thousands of entries) and the prefix has cut units next to whole ones and next
to units of empty lists; row thresholds that set aside none, some and most of a
cut unit's rows; level rows and counts against the oracle's vertex-level walk."""
import numpy as np
import pytest

import oracle
from gem_amd import GemContext, Graph, Query

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def case():
    g = Graph.rmat(10, 60.0, 4, 77)
    qs, refs, i = [], [], 0
    while len(qs) < 6:
        q = Query.random_walk(g, 3 + len(qs) % 2, 40 + i)
        i += 1
        if q.num_e >= 2:
            r = oracle.count(g, q)
            qs.append(q)
            refs.append(oracle.vcount(g, q, oracle.vertex_order_from_edges(q, r["order"])))
    return g, qs, refs


@pytest.mark.parametrize("blocks", [1, 48, 2048])
@pytest.mark.parametrize("heavy", [(1 << 20, 1024), (1024, 1024), (48, 64)])
def test_cut_units(case, blocks, heavy):
    g, qs, refs = case
    with GemContext(0) as ctx:
        ctx.load_data(g)
        ctx.set_persistent_blocks(blocks)
        ctx.set_heavy_split(*heavy)
        for q, r, ref in zip(qs, ctx.match_batch(qs), refs):
            assert r["count"] == ref["count"]
            assert np.array_equal(r["level_rows"], ref["level_rows"])


@pytest.mark.parametrize("blocks", [1, 2048])
@pytest.mark.parametrize("heavy", [(1024, 1024), (48, 64)])
def test_capped_final_walks(case, blocks, heavy):
    # under a cap that no query reaches, final levels are measured and walked in
    # runs of equal cost too
    g, qs, refs = case
    with GemContext(0) as ctx:
        ctx.load_data(g)
        ctx.set_persistent_blocks(blocks)
        ctx.set_heavy_split(*heavy)
        for graph in (False, True):
            ctx.set_graph(graph)
            for q, r, ref in zip(qs, ctx.match_batch(qs, cap=10 ** 8), refs):
                assert not r["saturated"] and r["count"] == ref["count"]
        for q, r, ref in zip(qs, ctx.match_batch(qs, cap=30000), refs):
            assert r["saturated"] == (ref["count"] > 30000)
            assert r["count"] == min(ref["count"], 30000)
