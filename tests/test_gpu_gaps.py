"""Graphs whose rows with ids lie far apart: long runs of empty rows between
them, which a tile of the row count, of the split count's transposition and of
its packing may span.  A vertex is moved up, in order, to where the run ends, so
the counts stay those of the graph without the runs."""
import numpy as np
import pytest

import oracle as O
import wtc

pytestmark = pytest.mark.gpu


def _spread(g, at, n):
    """g with vertex v moved to at[v] (ascending) of n."""
    rp = np.zeros(n + 1, dtype=np.uint64)
    rp[at + 1] = np.diff(g.row_ptr.astype(np.int64))
    np.cumsum(rp, out=rp)
    return wtc.CSR(n, g.m, rp, at[g.col_ind].astype(np.uint32))


def _complete(k):
    i, j = np.triu_indices(k, 1)
    return np.stack([i, j], axis=1)


def _graphs():
    r = np.random.default_rng(8)
    rmat = wtc.preprocess(wtc.gen_rmat(13, 16, seed=6))
    er = wtc.preprocess(wtc.gen_erdos_renyi(30000, 8 / 30000, seed=2))
    k300 = wtc.preprocess(wtc.graph_from_pairs(_complete(300).astype(np.uint32)))
    for name, g in (("rmat", rmat), ("er", er), ("K_300", k300)):
        v = np.arange(g.n)
        for gap in (1, 255, 256 * 16 - 1, 512 * 16, 1024 * 17 + 1, 1 << 20, 3000000):  # one run, before the last tenth
            at = v + gap * (v >= g.n - g.n // 10)
            yield f"{name} one run of {gap}", g, at, at[-1] + 1
        for step in (3, 40, 300):  # a run before every row
            if g.n * step < 6 << 20:
                yield f"{name} step {step}", g, v * step + step - 1, g.n * step + 100
        at = np.sort(r.choice(5 << 20, size=g.n, replace=False))  # runs of any length
        yield f"{name} anywhere", g, at, 5 << 20
        at = np.concatenate([v[:g.n // 2] * 200, g.n // 2 * 200 + 100000 + v[:g.n - g.n // 2]])  # sparse, then dense
        yield f"{name} sparse and dense", g, at, at[-1] + 5000


@pytest.mark.parametrize("ob", [4, 8])
def test_runs_of_empty_rows(gpu_ctx, ob):
    expect = {}
    try:
        for name, g, at, n in _graphs():
            if id(g) not in expect:
                expect[id(g)] = O.tc_merge(g)
            e, W = expect[id(g)], g.wedges()
            s = _spread(g, at, int(n))
            assert s.wedges() == W and s.validate_oriented(), name
            dg = gpu_ctx.upload(s, offset_bytes=ob)
            gpu_ctx.set_count_kernel(wtc.KERNEL_ROWS)
            cnt, st = dg.count(8, 0, stats=True)
            assert (cnt, st.wedges) == (e, W), name
            gpu_ctx.set_count_kernel(wtc.KERNEL_SPLIT)
            for a in (64, 8192, 1 << 20):
                cnt, st = dg.count(8, a, stats=True)
                assert (cnt, st.wedges, st.split) == (e, W, 1), (name, a)
                assert dg.count(8, a, 0, W // 3) + dg.count(8, a, W // 3, W) == e, (name, a)
            dg.free()
    finally:
        gpu_ctx.set_count_kernel(wtc.KERNEL_WALK)


def test_hubs_between_the_wedges(gpu_ctx):
    """Three million hubs of four leaves each, above every vertex of the triangles
    and below those of a core: their empty rows lie between the rows with
    wedges.  The staged kernel does not go by rows; twice its time is left to the
    row count (walked through window by window: fifteen times) and the split
    count has its time on the graph without most hubs and three times that."""
    def graph(hubs):
        o = 200 + 3 * np.arange(100000)
        h = 300200 + np.arange(hubs)
        leaves = 300200 + hubs + np.arange(4 * hubs)
        return wtc.DeviceGraph.from_pairs(gpu_ctx, np.concatenate([
            _complete(200), np.stack([o, o + 1], axis=1), np.stack([o, o + 2], axis=1), np.stack([o + 1, o + 2], axis=1),
            np.stack([np.repeat(h, 4), leaves], axis=1)]).astype(np.uint32))

    expect = 200 * 199 * 198 // 6 + 100000
    took = {}
    try:
        for hubs in (30000, 3000000):
            dg = graph(hubs)
            for kernel, a in ((wtc.KERNEL_STAGED, 0), (wtc.KERNEL_ROWS, 0), (wtc.KERNEL_SPLIT, 4096)):
                gpu_ctx.set_count_kernel(kernel)
                ms = []
                for _ in range(6):
                    cnt, st = dg.count(8, a, stats=True)
                    assert cnt == expect and st.split == (kernel == wtc.KERNEL_SPLIT)
                    ms.append(st.prefix_ms + st.bitmap_ms + st.count_ms)
                took[hubs, kernel] = min(ms)
            dg.free()
    finally:
        gpu_ctx.set_count_kernel(wtc.KERNEL_WALK)
    print(took)
    assert took[3000000, wtc.KERNEL_ROWS] < 2 * took[3000000, wtc.KERNEL_STAGED], took
    assert took[3000000, wtc.KERNEL_SPLIT] < 4 * took[30000, wtc.KERNEL_SPLIT], took
