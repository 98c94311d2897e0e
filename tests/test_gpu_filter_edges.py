"""GPU: the filter where its kernels hand over: degrees around the one-lane and
one-wave limits, a hub of several counting rounds, a ragged last tile and more
than one rank chunk, labels in bytes and in words, thresholds 0 and 1; candidate
lists and positions bit-equal to the oracle's."""
import numpy as np
import pytest

import oracle
from gem_amd import GemContext, Graph, Query

pytestmark = pytest.mark.gpu

N = 270017  # 4,220 tiles: two chunks of ranks, the last tile of 1 vertex


def _graph(num_labels):
    rng = np.random.default_rng(num_labels)
    pairs = [rng.integers(100, N, (300000, 2))]
    for h, deg in enumerate((63, 64, 65, 127, 128, 4095, 4096, 4097, 9000, 130000)):
        pairs.append(np.stack([np.full(deg, h), rng.choice(np.arange(100, N), deg, replace=False)], 1))
    e = np.concatenate(pairs)
    e = e[e[:, 0] != e[:, 1]]
    e = np.unique(np.sort(e, 1), axis=0)
    labels = rng.integers(0, num_labels, N).astype(np.uint32)
    labels[:10] = 1
    return Graph.from_edges(N, e, labels)


def _queries(num_labels):
    lab = np.array([1, 0, 2, 1, 0], np.uint32)
    yield Query(lab, np.array([[0, 1], [0, 2], [0, 3], [1, 2], [3, 4]]))
    # 20 vertices, so that several label slots and counts past one occur
    k = np.arange(20)
    yield Query((k % min(num_labels, 7)).astype(np.uint32), np.stack([k[:-1] // 2, k[1:]], 1))


@pytest.mark.parametrize("num_labels", [3, 300])
def test_candidates_and_positions(num_labels):
    g = _graph(num_labels)
    with GemContext(0) as ctx:
        ctx.load_data(g)
        for q in _queries(num_labels):
            for t in (0, 1):
                num, lists = ctx.filter(q, threshold=t)
                ref = oracle.filter(g, q, threshold=t)
                for u in range(q.num_v):
                    assert np.array_equal(lists[u], ref[u])
                probe = np.concatenate([np.arange(10), [N - 1], lists[0][-3:]]).astype(np.uint32)
                want = np.searchsorted(lists[0], probe)
                hit = np.isin(probe, lists[0])
                assert np.array_equal(ctx.position_lookup(0, probe), np.where(hit, want, 0xFFFFFFFF))


@pytest.mark.parametrize("num_labels", [3, 300])
def test_edge_tables(num_labels):
    """Offsets and values over several scan chunks (lists past 4,096
    candidates) and rows of one to 64 pieces."""
    g = _graph(num_labels)
    with GemContext(0) as ctx:
        ctx.load_data(g)
        q = next(_queries(num_labels))
        num, _ = ctx.filter(q, want_lists=False)
        sizes = ctx.build_edge_tables()
        assert np.array_equal(sizes, oracle.table_sizes(g, q))
        for d in range(2 * q.num_e):
            u = int(q.edges[d // 2][d % 2])
            ref = oracle.edge_table(g, q, d, int(num[u]), int(sizes[d]))
            if ref is None:  # keyed on a leaf
                assert sizes[d] == 0
                continue
            off, val = ctx.read_edge_table(d, int(num[u]), int(sizes[d]))
            assert np.array_equal(off, ref[0]) and np.array_equal(val, ref[2])
