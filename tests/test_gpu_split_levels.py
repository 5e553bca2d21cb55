"""GPU split count where the transposition's shape changes: key counts on
both sides of every part size, two and three levels, in-edge tiles that end
inside rows and cross long runs of vertices without in-edges, and tiles of
the row kernel over rows with no, one and many in-edges."""
import numpy as np
import pytest

import oracle as O
import wtc

pytestmark = pytest.mark.gpu

SLAB = 2048  # colInd positions per list key


@pytest.fixture
def split_ctx(gpu_ctx):
    gpu_ctx.set_count_kernel(wtc.KERNEL_SPLIT)
    try:
        yield gpu_ctx
    finally:
        gpu_ctx.set_count_kernel(wtc.KERNEL_WALK)


def _check(ctx, g, a, expect, ob=4):
    dg = ctx.upload(g, offset_bytes=ob)
    try:
        W = g.wedges()
        cnt, st = dg.count(4, a, stats=True)
        assert cnt == expect and st.split == 1 and st.wedges == W, a
        cuts = [0, W // 3, W // 3 + 1, W - W // 5, W]
        parts = [dg.count(4, a, lo, hi) for lo, hi in zip(cuts, cuts[1:])]
        assert sum(parts) == expect, (a, parts)
    finally:
        dg.free()


@pytest.mark.parametrize("ob,narrow", [(4, "1"), (8, "0")])
def test_key_counts_around_part_sizes(split_ctx, monkeypatch, ob, narrow):
    """2^16, 2^17 and 2^19 keys, one row group of 32 below and above: parts of
    256 to 2,048 keys grouped in two levels, and three levels past 2^19."""
    monkeypatch.setenv("WTC_SPLIT_NARROW", narrow)
    rng = np.random.default_rng(3)
    n = 1 << 20
    hubs = rng.integers(0, 400, size=(60000, 2))
    flat = rng.integers(0, n, size=(400000, 2))
    mixed = np.stack([rng.integers(0, 400, 200000), rng.integers(0, n, 200000)], axis=1)
    g = wtc.preprocess(wtc.graph_from_pairs(np.concatenate([hubs, flat, mixed]).astype(np.uint32)))
    expect = O.tc_merge(g)
    slabs = (g.m + SLAB - 1) // SLAB
    for keys in (1 << 16, 1 << 17, 1 << 19):
        edge = (keys - slabs) // 32 * 32  # the last a with at most that many keys
        for a in (edge, edge + 32):
            if 0 < a <= (g.n + 31) // 32 * 32:
                _check(split_ctx, g, a, expect, ob)


@pytest.mark.parametrize("tail", [0, 1, 4095, 4096, 4097, 9000])
def test_in_edge_tiles(split_ctx, tail):
    """In-edge counts just below, at and above the tiles of 4,096, with
    thousands of vertices without in-edges before, between and after."""
    k = 40
    i, j = np.triu_indices(k, 1)
    base = 20000
    pairs = [np.stack([base + 3 * i, base + 3 * j], axis=1)]  # K_40 on every third id
    # `tail` disjoint triangles, one in-edge each, on ids past a gap
    t = np.arange(tail)
    b = base + 1000 + 5 * t
    for x, y in ((0, 1), (0, 2), (1, 2)):
        pairs.append(np.stack([b + x, b + y], axis=1))
    g = wtc.preprocess(wtc.graph_from_pairs(np.concatenate(pairs).astype(np.uint32)))
    expect = k * (k - 1) * (k - 2) // 6 + tail
    for a in (32, 64, (g.n + 31) // 32 * 32):
        _check(split_ctx, g, a, expect)


def test_rows_with_few_in_edges(split_ctx):
    """A row with thousands of in-edges among rows with one and none: tiles of
    the row kernel that start and end inside a row and inside a row's fixed
    share of the work."""
    rng = np.random.default_rng(8)
    m = 30000
    leaf = 10 + np.arange(m)
    pairs = [np.stack([np.zeros(m, np.int64), leaf], axis=1), np.stack([np.ones(m, np.int64), leaf], axis=1),
             np.array([[0, 1]])]
    extra = rng.integers(10, 10 + m, size=(5000, 2))
    g = wtc.preprocess(wtc.graph_from_pairs(np.concatenate(pairs + [extra]).astype(np.uint32)))
    expect = O.tc_merge(g)
    for a in (32, 4096, (g.n + 31) // 32 * 32):
        _check(split_ctx, g, a, expect)
