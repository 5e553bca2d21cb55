"""GPU split count with nearly every wedge in its list part: rows of every
length up to the longest hashed and past it, whose ids lie at random among
other rows' so that their hash sets have full buckets, and short tails and
long ones (four and eight lanes to a tail)."""
import numpy as np
import pytest

import wtc

pytestmark = pytest.mark.gpu


def _cliques(count, k, seed):
    """`count` cliques of k vertices whose ranks interleave at random: each
    vertex has up to 200 leaves."""
    rng = np.random.default_rng(seed)
    i, j = np.triu_indices(k, 1)
    pairs = [np.stack([c * k + i, c * k + j], axis=1) for c in range(count)]
    leaves = np.repeat(np.arange(count * k), rng.integers(0, 200, count * k))
    pairs.append(np.stack([leaves, count * k + np.arange(leaves.size)], axis=1))
    return wtc.preprocess(wtc.graph_from_pairs(np.concatenate(pairs).astype(np.uint32)))


@pytest.mark.parametrize("count,k", [(8, 1030), (300, 20)])
@pytest.mark.parametrize("ob,narrow", [(4, "1"), (8, "0")])
def test_interleaved_cliques(gpu_ctx, monkeypatch, count, k, ob, narrow):
    monkeypatch.setenv("WTC_SPLIT_NARROW", narrow)
    g = _cliques(count, k, 9)
    expect = count * k * (k - 1) * (k - 2) // 6
    gpu_ctx.set_count_kernel(wtc.KERNEL_SPLIT)
    dg = gpu_ctx.upload(g, offset_bytes=ob)
    try:
        W = g.wedges()
        cnt, st = dg.count(4, 32, stats=True)
        assert cnt == expect and st.split == 1
        if k > 1000:
            assert st.list_in_edges > 0.9 * (st.list_in_edges + st.in_edges)
        cuts = [0, W // 3, W // 3 + 1, W - W // 5, W]
        assert sum(dg.count(4, 32, lo, hi) for lo, hi in zip(cuts, cuts[1:])) == expect
    finally:
        dg.free()
        gpu_ctx.set_count_kernel(wtc.KERNEL_WALK)


@pytest.mark.parametrize("ob,narrow", [(4, "1"), (8, "0")])
def test_rows_past_the_longest_hashed(gpu_ctx, monkeypatch, ob, narrow):
    """A quarter of the rows too long for a hash set: searched, four ids of a
    tail side by side, with tails of every length and alignment."""
    monkeypatch.setenv("WTC_SPLIT_NARROW", narrow)
    count, k = 12, 1400
    g = _cliques(count, k, 11)
    expect = count * k * (k - 1) * (k - 2) // 6
    gpu_ctx.set_count_kernel(wtc.KERNEL_SPLIT)
    dg = gpu_ctx.upload(g, offset_bytes=ob)
    try:
        cnt, st = dg.count(4, 32, stats=True)
        assert cnt == expect and st.split == 1 and st.list_in_edges > st.in_edges
    finally:
        dg.free()
        gpu_ctx.set_count_kernel(wtc.KERNEL_WALK)
