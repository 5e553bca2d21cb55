"""GPU row count (KERNEL_ROWS): edges against hashed rows, at the sizes of its
tiles, lists and rows, alone and in sets, against closed forms and the
oracle."""
import numpy as np
import pytest

import oracle as O
import wtc

pytestmark = pytest.mark.gpu


@pytest.fixture
def rows_ctx(gpu_ctx):
    gpu_ctx.set_count_kernel(wtc.KERNEL_ROWS)
    try:
        yield gpu_ctx
    finally:
        gpu_ctx.set_count_kernel(wtc.KERNEL_WALK)


def _complete(k, first=0):
    i, j = np.triu_indices(k, 1)
    return np.stack([first + i, first + j], axis=1)


def _graph(*pairs):
    p = np.concatenate(pairs) if pairs else np.zeros((0, 2))
    return wtc.preprocess(wtc.graph_from_pairs(p.astype(np.uint32)))


def _graphs():
    rng = np.random.default_rng(4)
    yield "no edges", _graph()
    yield "one edge", _graph(np.array([[0, 1]]))
    yield "path", _graph(np.stack([np.arange(2000), np.arange(2000) + 1], axis=1))
    yield "star", _graph(np.stack([np.zeros(3000, int), 1 + np.arange(3000)], axis=1))
    for k in (3, 17, 18, 33, 65, 66, 129, 140):  # lists of up to 16 and 64 ids, and longer ones
        yield f"K_{k}", _graph(_complete(k))
    yield "gaps", _graph(*[_complete(5, 4000 * b) for b in range(30)])  # long runs of vertices without edges
    for k in (512, 513, 514, 700, 1100):  # rows up to, just over and far over the longest hashed
        yield f"K_{k}", _graph(_complete(k))
    yield "er", wtc.preprocess(wtc.gen_erdos_renyi(3000, 0.01, seed=3))
    yield "ba", wtc.preprocess(wtc.gen_barabasi_albert(4000, 9, seed=5))
    yield "rmat", wtc.preprocess(wtc.gen_rmat(13, 16, seed=6))
    # hubs of several hundred neighbours whose rows cross tiles
    hubs = np.stack([rng.integers(0, 600, 90000), rng.integers(0, 900, 90000)], axis=1)
    yield "hubs", _graph(hubs, rng.integers(0, 20000, size=(30000, 2)))


@pytest.mark.parametrize("ob", [4, 8])
def test_rows_match_oracle(rows_ctx, ob):
    for name, g in _graphs():
        expect = O.tc_merge(g)
        dg = rows_ctx.upload(g, offset_bytes=ob)
        for s, a in ((1, 0), (8, 64)):
            cnt, st = dg.count(s, a, stats=True)
            assert cnt == expect and st.wedges == g.wedges() and st.split == 0, (name, s, a)
        W = g.wedges()
        if W > 3:  # ranges take another kernel and still add up
            assert dg.count(4, 0, 0, W // 3) + dg.count(4, 0, W // 3, W) == expect, name
        dg.free()


def test_rows_in_sets(rows_ctx):
    """Sets: tiles found across graphs, empty ones among them, colInd starts
    on any element, replays and host batches; the small-graph kernel off."""
    cur, _ = rows_ctx.small_graphs()
    graphs = [g for _, g in _graphs()]
    expect = [O.tc_merge(g) for g in graphs]
    try:
        rows_ctx.set_small_graphs(0)
        b = wtc.Batch(rows_ctx, graphs)
        for _ in range(3):
            got, st = b.count(stats=True)
            assert got.tolist() == expect and st.wedges == sum(g.wedges() for g in graphs)
            wtc.tc_gpu(graphs[7], 4, 0)  # eager work between replays
        b.free()
        got, st = wtc.batch_count_host(rows_ctx, graphs, stats=True)
        assert got.tolist() == expect and st.wedges == sum(g.wedges() for g in graphs)
        many = [graphs[i % 6 + 4] for i in range(150)]  # more graphs than a kernel fetches itself
        assert wtc.batch_count_host(rows_ctx, many).tolist() == [expect[i % 6 + 4] for i in range(150)]
    finally:
        rows_ctx.set_small_graphs(cur)
