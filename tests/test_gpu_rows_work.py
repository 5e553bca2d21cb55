"""GPU row count where an edge's adj+(w) is long and what is left of v's row is
short, where a row is longer than a tile, and the work of a graph of a dense
core with many members of few neighbours."""
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


def _complete(k):
    i, j = np.triu_indices(k, 1)
    return np.stack([i, j], axis=1)


def _core_and_members(k, ids):
    """K_k and a vertex for each row of ids, joined to those of the core."""
    v = k + np.arange(len(ids))
    pairs = [_complete(k)] + [np.stack([v, ids[:, i]], axis=1) for i in range(ids.shape[1])]
    return wtc.preprocess(wtc.graph_from_pairs(np.concatenate(pairs).astype(np.uint32)))


def _csr(rows, n):
    """An oriented CSR of the rows given (vertex: its ids), not ordered by degree."""
    d = np.zeros(n, dtype=np.uint64)
    for v, x in rows.items():
        d[v] = len(x)
    rp = np.zeros(n + 1, dtype=np.uint64)
    np.cumsum(d, out=rp[1:])
    col = np.concatenate([np.sort(rows[v]) for v in sorted(rows)]).astype(np.uint32)
    return wtc.CSR(n, int(rp[n]), rp, col)


def _graphs():
    r = np.random.default_rng(3)
    # every length of adj+(w) up to 149 with one id left after w, and up to 199 with one to five
    yield "pairs", _core_and_members(150, _complete(150))
    for k in (3, 4, 5, 6):
        yield f"{k} each", _core_and_members(200, np.sort(np.stack([r.permutation(200)[:k] for _ in range(6000)]), axis=1))
    # rows to the longest hashed and over it, beginning anywhere in a tile
    for longest in (513, 1025, 2047, 2048, 2049, 2600):
        n = 9000
        rows = {0: 1 + np.arange(r.integers(1, 500)), 1: 2 + np.arange(longest)}
        for w in r.permutation(np.arange(2, 2 + longest))[:400]:
            size = int(r.choice([1, 7, 40, 300, 2500, 5000]))
            rows[int(w)] = r.choice(np.arange(w + 1, n), size=min(size, n - 1 - w), replace=False)
        yield f"row of {longest}", _csr(rows, n)


@pytest.mark.parametrize("ob", [4, 8])
def test_short_tails_and_long_rows(rows_ctx, ob):
    graphs = list(_graphs())
    expect = [O.tc_merge(g) for _, g in graphs]
    for (name, g), e in zip(graphs, expect):
        assert g.validate_oriented()
        dg = rows_ctx.upload(g, offset_bytes=ob)
        cnt, st = dg.count(8, 0, stats=True)
        assert cnt == e and st.wedges == g.wedges(), name
        dg.free()
    if ob == 4:  # as a set: rows begin at other places of their tiles
        b = wtc.Batch(rows_ctx, [g for _, g in graphs])
        assert b.count().tolist() == expect
        b.free()


def test_complete_graphs_of_long_rows(rows_ctx):
    for k in (2048, 2049, 2050, 2300):  # rows of up to 2,048 ids are hashed
        dg = wtc.DeviceGraph.from_pairs(rows_ctx, _complete(k).astype(np.uint32))
        assert dg.count(8, 0) == k * (k - 1) * (k - 2) // 6
        dg.free()


def test_members_of_a_core_cost_no_more_than_by_the_staged_kernel(gpu_ctx):
    """1,000 vertices all joined and two million of two neighbours among them:
    twice the staged kernel's time is left to the row count, which streaming
    every adj+(w) would take more than four times."""
    r = np.random.default_rng(1)
    first = r.integers(0, 1000, 2000000)
    ids = np.stack([first, (first + r.integers(1, 500, 2000000)) % 1000], axis=1)
    v = 1000 + np.arange(len(ids))
    pairs = np.concatenate([_complete(1000)] + [np.stack([v, ids[:, i]], axis=1) for i in range(2)]).astype(np.uint32)
    dg = wtc.DeviceGraph.from_pairs(gpu_ctx, pairs)
    took, counts = {}, set()
    try:
        for kernel, a in ((wtc.KERNEL_STAGED, 2048), (wtc.KERNEL_ROWS, 0)):
            gpu_ctx.set_count_kernel(kernel)
            ms = []
            for _ in range(6):
                cnt, st = dg.count(4, a, stats=True)
                counts.add(cnt)
                ms.append(st.prefix_ms + st.bitmap_ms + st.count_ms)
            took[kernel] = min(ms)
    finally:
        gpu_ctx.set_count_kernel(wtc.KERNEL_WALK)
        dg.free()
    assert counts == {1000 * 999 * 998 // 6 + 2000000}
    assert took[wtc.KERNEL_ROWS] < 2 * took[wtc.KERNEL_STAGED], took
