"""GPU split count around the packed copy of the top ids: bitmap lengths on
both sides of the nearest 65,528 ranks and of every field width past them,
rows of every small length with ids on both sides of that line, and wedge
ranges that cut one tail at the front, at the end and at both."""
import numpy as np
import pytest

import oracle as O
import wtc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cliques():
    """Cliques of 3 to 40 random vertices among 600,000, each vertex in about
    one: rows of 0 to some 80 ids all over the ranks."""
    rng = np.random.default_rng(5)
    pairs = []
    for k in [3, 4, 5, 8, 9, 15, 16, 17, 18, 25, 40] * 3000:
        v = rng.integers(0, 600000, k)
        i, j = np.triu_indices(k, 1)
        pairs.append(np.stack([v[i], v[j]], axis=1))
    g = wtc.preprocess(wtc.graph_from_pairs(np.concatenate(pairs).astype(np.uint32)))
    assert g.n > 1 << 18
    return g, O.tc_merge(g)


@pytest.mark.parametrize("ob,narrow", [(4, "1"), (8, "0")])
def test_bitmap_lengths_around_the_layouts(gpu_ctx, monkeypatch, cliques, ob, narrow):
    monkeypatch.setenv("WTC_SPLIT_NARROW", narrow)
    g, expect = cliques
    gpu_ctx.set_count_kernel(wtc.KERNEL_SPLIT)
    dg = gpu_ctx.upload(g, offset_bytes=ob)
    try:
        W = g.wedges()
        top = (g.n + 31) // 32 * 32
        for a in (65504, 65536, 65568, 131072, 262144, 262176, top):
            if a > top:
                continue
            cnt, st = dg.count(4, a, stats=True)
            assert cnt == expect and st.split == 1, a
            assert st.in_edges + st.list_in_edges <= g.m and st.top_wedges <= W, a
        # all tails of one row and more, cut one wedge apart
        a, mid = 131072, W // 2
        cuts = [0, 1, 2, 3, mid, *range(mid + 1, mid + 40), W - 2, W - 1, W]
        parts = [dg.count(4, a, lo, hi) for lo, hi in zip(cuts, cuts[1:])]
        assert sum(parts) == expect and max(parts[:3]) <= 1, parts
    finally:
        dg.free()
        gpu_ctx.set_count_kernel(wtc.KERNEL_WALK)
