"""GPU: expansions fused with the selects after them against the stepwise join
(which profiling takes) and the oracle.

Dense graphs of one and two labels (equal-label columns), queries whose
expansions are followed by one to three selects, keyed by old and by new columns,
in the middle and at the end; whole levels and levels cut by a small budget, with
and without caps and work limits, where the rows processed must be the same."""
import numpy as np
import pytest

import oracle
from gem_amd import GemContext, Graph, Query

pytestmark = pytest.mark.gpu

CLIQUE = {k: [(a, b) for b in range(k) for a in range(b)] for k in (3, 4, 5)}
SHAPES = {
    "triangle": (3, CLIQUE[3]),
    "clique4": (4, CLIQUE[4]),
    "clique5": (5, CLIQUE[5]),
    "square": (4, [(0, 1), (1, 2), (2, 3), (0, 3)]),
    "diamond_tail": (5, CLIQUE[4][:5] + [(3, 4)]),
    "clique4_tail": (5, CLIQUE[4] + [(0, 4)]),
}


def _graph(scale, deg, labels):
    return Graph.rmat(scale, deg, labels, 31)


@pytest.mark.parametrize("shape", sorted(SHAPES))
@pytest.mark.parametrize("labels,scale,deg", [(1, 9, 10.0), (2, 10, 24.0)])
@pytest.mark.parametrize("budget", [1 << 33, 1 << 20])
def test_fused_equals_steps(shape, labels, scale, deg, budget):
    g = _graph(scale, deg, labels)
    nv, edges = SHAPES[shape]
    q = Query((np.arange(nv) % labels).astype(np.uint32), np.array(edges))
    with GemContext(0) as ctx:
        ctx.load_data(g)
        ctx.set_level_budget(budget)

        def both(cap=0):
            got = ctx.match_full(q, cap=cap)
            ctx.set_profiling(True)
            steps = ctx.match_full(q, cap=cap)
            ctx.set_profiling(False)
            assert all(got[x] == steps[x] for x in ("count", "saturated", "work_limited", "rows_processed"))
            return got

        r = both()
        if r["count"] < 10 ** 6:
            assert r["count"] == oracle.count(g, q)["count"]
        for cap in {1, max(1, r["count"] // 2), r["count"] + 1}:
            both(cap)
        for limit in (r["rows_processed"] // 2, r["rows_processed"] - 1, r["rows_processed"]):
            ctx.set_work_limit(max(1, limit))
            assert both()["work_limited"] == (limit < r["rows_processed"])
