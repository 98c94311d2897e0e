"""GPU: the filter and table times of a batch are both those of its last group
of queries prepared together."""
import pytest

from gem_amd import GemContext, Graph, Query

pytestmark = pytest.mark.gpu


def test_batch_times_cover_the_group():
    """A batch of 32 equal queries takes both phases 32 times as much device work
    as a batch of one: a quarter of that is asked for."""
    g = Graph.rmat(17, 16.0, 8, 5)
    q = Query.random_walk(g, 6, 3)
    with GemContext(0) as ctx:
        ctx.load_data(g)
        ms = {}
        for n in (1, 32):
            for _ in range(3):  # the fastest of three
                ctx.match_batch([q] * n, cap=1)
                t = ctx.phase_times()
                ms[n] = [min(a, b) for a, b in zip(ms.get(n, (1e9, 1e9)), (t["filter_ms"], t["tables_ms"]))]
        assert ms[32][0] > 8 * ms[1][0] > 0
        assert ms[32][1] > 8 * ms[1][1] > 0
