"""GPU split count: the dense part (wedges among the last ranks as a product
of bit matrices), around its tile and class sizes, against closed forms and
the oracle."""
import numpy as np
import pytest

import oracle as O
import wtc

pytestmark = pytest.mark.gpu


@pytest.fixture
def split_ctx(gpu_ctx):
    gpu_ctx.set_count_kernel(wtc.KERNEL_SPLIT)
    try:
        yield gpu_ctx
    finally:
        gpu_ctx.set_count_kernel(wtc.KERNEL_WALK)


def _complete(k, pad=0):
    i, j = np.triu_indices(k, 1)
    p = np.stack([i, j], axis=1)
    if pad:  # a path of `pad` low-degree vertices, ranked before the clique
        x = k + np.arange(pad)
        p = np.concatenate([p, np.stack([x, x + 1], axis=1)])
    return wtc.preprocess(wtc.graph_from_pairs(p.astype(np.uint32)))


@pytest.mark.parametrize("k", [17, 33, 127, 128, 129, 255, 257, 511, 512, 513, 640, 1023, 1025, 2049])
def test_complete_graphs(split_ctx, k):
    """K_k, alone and behind a long path: class sizes, row tiles and core
    groups with one row or column to spare or missing, every wedge closed,
    whole and in ranges whose end vertices keep out of the dense part."""
    for pad in (0, 20000):
        g = _complete(k, pad)
        W = g.wedges()
        T = k * (k - 1) * (k - 2) // 6
        dg = split_ctx.upload(g)
        for a in (32, 512, (g.n + 31) // 32 * 32):
            cnt, st = dg.count(4, a, stats=True)
            assert cnt == T and st.split == 1 and st.wedges == W, (pad, a)
            dense_w, dense_e = split_ctx.debug_split()
            assert dense_w <= st.top_wedges and dense_e <= st.in_edges
            cuts = [0, W // 5, W // 2, W // 2 + 1, W]
            assert sum(dg.count(4, a, lo, hi) for lo, hi in zip(cuts, cuts[1:])) == T, (pad, a)
        dg.free()


@pytest.mark.parametrize("ob,narrow", [(4, "1"), (8, "1"), (8, "0")])
def test_planted_cores(split_ctx, monkeypatch, ob, narrow):
    """A random graph whose last ranks hold cores of several densities, so
    that several classes are in use at once and rows sit on both sides of
    the class limits: the oracle's count, and the dense part takes wedges."""
    monkeypatch.setenv("WTC_SPLIT_NARROW", narrow)
    rng = np.random.default_rng(21)
    n = 40000
    parts = [rng.integers(0, n, size=(150000, 2))]
    for size, edges in ((300, 30000), (1500, 150000), (6000, 500000)):
        parts.append(rng.integers(0, size, size=(edges, 2)))
    hubs = rng.integers(0, 400, size=60000)  # rows with many ids among the last ranks, far below them
    parts.append(np.stack([hubs, 6000 + rng.integers(0, 1000, size=60000)], axis=1))
    g = wtc.preprocess(wtc.graph_from_pairs(np.concatenate(parts).astype(np.uint32)))
    expect = O.tc_merge(g)
    W = g.wedges()
    dg = split_ctx.upload(g, offset_bytes=ob)
    for a in (64, 4096, 16384):
        cnt, st = dg.count(8, a, stats=True)
        assert cnt == expect and st.split == 1
        assert split_ctx.debug_split()[0] > 0
        lo, hi = W // 4, W // 4 + W // 300
        assert dg.count(8, a, lo, hi) == O.tc_wedge(g, 8, a, lo, hi)
    dg.free()
