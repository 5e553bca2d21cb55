"""The split count of a graph of more than 2^31 vertices, whose ids leave its
hash sets no bit to mark a full bucket with.  About 60 GB of device memory and 40
GB of the host's."""
import numpy as np
import pytest

import oracle as O
import wtc

pytestmark = pytest.mark.gpu


def _complete(k):
    i, j = np.triu_indices(k, 1)
    return np.stack([i, j], axis=1)


def test_split_count_of_ids_above_31_bits():
    r = np.random.default_rng(12)
    hubs = np.stack([r.integers(0, 900, 60000), r.integers(0, 30000, 60000)], axis=1)
    g = wtc.preprocess(wtc.graph_from_pairs(np.concatenate([_complete(280), hubs]).astype(np.uint32)))
    expect, W = O.tc_merge(g), g.wedges()
    # some vertices in front, the others across 2^31 in steps
    front = 50
    at = np.concatenate([np.arange(front), (1 << 31) - 3000 + 7 * np.arange(g.n - front)])
    n = int(at[-1]) + 1
    assert n > (1 << 31) + 100000
    rp = np.zeros(n + 1, dtype=np.uint64)
    rp[at + 1] = np.diff(g.row_ptr.astype(np.int64))
    np.cumsum(rp, out=rp)
    s = wtc.CSR(n, g.m, rp, at[g.col_ind].astype(np.uint32))
    ctx = wtc.Context(0)
    dg = ctx.upload(s, offset_bytes=4)
    del s, rp
    ctx.set_count_kernel(wtc.KERNEL_SPLIT)
    for a in (64, 65536, 1 << 20):  # list rows only, both, top rows only
        cnt, st = dg.count(8, a, stats=True)
        assert (cnt, st.wedges, st.split) == (expect, W, 1), a
        assert dg.count(8, a, 0, W // 3) + dg.count(8, a, W // 3, W) == expect, a
    ctx.set_count_kernel(wtc.KERNEL_WALK)
    assert dg.count(8, 64) == expect
    dg.free()
    ctx.close()
