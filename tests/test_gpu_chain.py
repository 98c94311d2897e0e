"""GPU: the plain join's chained steps against the stepwise ones (a log is
asked for there) and the oracle: levels below, at the switch, and above the
chain's room, small level budgets, empty levels, caps and work limits."""
import numpy as np
import pytest

import oracle
from gem_amd import GemContext, Graph, Query

pytestmark = pytest.mark.gpu


def _star(n, leaves):
    """A hub joined to `leaves` vertices of one label: levels of leaves^k rows."""
    e = np.stack([np.zeros(leaves, np.int64), np.arange(1, leaves + 1)], 1)
    lab = np.ones(n, np.uint32)
    lab[0] = 0
    return Graph.from_edges(n, e, lab)


@pytest.mark.parametrize("leaves", [3, 65, 511, 513])
def test_star_levels(leaves):
    # 511 * 510 rows stay below 2^18, 513 * 512 pass it
    g = _star(leaves + 2, leaves)
    q = Query(np.array([0, 1, 1, 1], np.uint32), np.array([[0, 1], [0, 2], [0, 3]]))
    want = leaves * (leaves - 1) * (leaves - 2)
    with GemContext(0) as ctx:
        ctx.load_data(g)
        for cap in (0, 1, want - 1, want):
            r = ctx.match_full(q, cap=cap)
            sat = bool(cap) and want > cap
            assert (r["count"], r["saturated"]) == (cap if sat else want, sat)
        rows = r["rows_processed"]
        ctx.set_work_limit(rows)
        assert ctx.match_full(q)["count"] == want
        ctx.set_work_limit(rows - 1)
        assert ctx.match_full(q)["work_limited"]


@pytest.mark.parametrize("scale,budget", [(10, 1 << 31), (12, 1 << 31), (12, 1 << 20)])
def test_chain_equals_steps(scale, budget):
    g = Graph.rmat(scale, 12.0, 4, 99)
    with GemContext(0) as ctx:
        ctx.load_data(g)
        ctx.set_level_budget(budget)
        for i in range(10):
            q = Query.random_walk(g, 3 + i % 4, 500 + i)
            if q.num_e < 2:
                continue
            r = ctx.match_full(q, cap=10 ** 7)
            logged = ctx.join(r["order"], cap=10 ** 7, log=True)
            assert (r["count"], r["saturated"]) == (logged["count"], logged["saturated"])
            ref = oracle.count(g, q, cap=10 ** 7)
            assert (r["count"], r["saturated"]) == (ref["count"], ref["saturated"])
        # no candidate of the second label: the first level is empty
        none = Query(np.array([0, 9, 0], np.uint32), np.array([[0, 1], [1, 2]]))
        assert ctx.match_full(none)["count"] == 0
