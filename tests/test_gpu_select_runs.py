"""GPU: where the fused expansion of the counting join hands over: more selects
after an expansion than one launch takes (the rest go on as steps of their own,
at the end and in the middle), and more equal-label columns than it has room for
(expansion and selects as steps).  The step log takes the steps one by one: its
rows say that the expansion is past the chained levels, and the counts of both,
and the oracle's, are the same."""
import numpy as np
import pytest

import oracle
from gem_amd import GemContext, Graph, Query

pytestmark = pytest.mark.gpu

CHAINED = 1 << 18  # rows up to which levels are chained


def _dense():
    rng = np.random.default_rng(5)
    return Graph.from_edges(60, np.argwhere(np.triu(rng.random((60, 60)) < 0.5, 1)), np.zeros(60, np.uint32))


def _ladder(m=60):
    """A closed ladder with a diagonal in every sixth square: few closed walks
    among millions of paths."""
    i = np.arange(m)
    e = np.concatenate([np.stack(x, 1) for x in ((i, (i + 1) % m), (m + i, m + (i + 1) % m), (i, m + i))])
    d = i[::6]
    e = np.concatenate([e, np.stack([d, m + (d + 1) % m], 1)])
    return Graph.from_edges(2 * m, np.unique(np.sort(e, 1), axis=0), np.zeros(2 * m, np.uint32))


def _clique(k, tail):
    e = [(a, b) for b in range(k) for a in range(b)] + ([(0, k)] if tail else [])
    return Query(np.zeros(k + tail, np.uint32), np.array(e))


def _cycle(k):
    return Query(np.zeros(k, np.uint32), np.array([(i, i + 1) for i in range(k - 1)] + [(0, k - 1)]))


def _check(g, q, step):
    """Edges in order; step = the expansion that has to be past the chain."""
    with GemContext(0) as ctx:
        ctx.load_data(g)
        ctx.filter(q, want_lists=False)
        ctx.build_edge_tables()
        order = np.arange(q.num_e)
        fused = ctx.join(order)
        steps = ctx.join(order, log=True)
        assert not steps["step_select"][step] and steps["step_rows"][step] > CHAINED
        assert fused["count"] == steps["count"] == oracle.vcount(g, q, np.arange(q.num_v))["count"] > 0
        return steps


@pytest.mark.parametrize("tail", [0, 1])
@pytest.mark.parametrize("k", [6, 7])  # four and five selects after the last vertex
def test_selects_of_one_expansion(k, tail):
    last = (k - 1) * (k - 2) // 2  # the expansion to vertex k - 1
    steps = _check(_dense(), _clique(k, tail), last)
    assert steps["step_select"][last + 1:last + k - 1].all()


@pytest.mark.parametrize("k", [16, 17, 18, 19])
def test_equal_label_columns(k):
    steps = _check(_ladder(), _cycle(k), k - 2)
    assert steps["step_select"][k - 1]
