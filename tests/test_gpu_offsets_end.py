"""Counts of a graph whose 4-byte row offsets end just below 2^32: every
kernel's positions in colInd reach it, and none may be stepped past it in 32
bits.  Vertex v of the graph is joined to the K after it, so every wedge is
closed and the counts are known; some vertices without edges come last.  About
140 GB of device memory and 40 GB of the host's."""
import gc
import time
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

import wtc

pytestmark = pytest.mark.gpu

K, ALONE = 46, 96


def _band(m_end):
    """The largest such graph of fewer than m_end edges, and its wedges."""
    n = (m_end - 1 + K * (K + 1) // 2) // K
    d = np.minimum(K, n - 1 - np.arange(n))
    rp = np.zeros(n + ALONE + 1, dtype=np.uint64)
    np.cumsum(d, out=rp[1:n + 1])
    rp[n + 1:] = rp[n]
    m = int(rp[n])
    col = np.empty(m, dtype=np.uint32)
    full = n - K  # rows of K ids

    def fill(v0):
        v1 = min(v0 + (1 << 20), full)
        col[v0 * K:v1 * K].reshape(-1, K)[:] = np.arange(v0, v1, dtype=np.uint32)[:, None] + np.arange(1, K + 1, dtype=np.uint32)

    with ThreadPoolExecutor(16) as ex:
        list(ex.map(fill, range(0, full, 1 << 20)))
    for v in range(full, n):
        col[int(rp[v]):int(rp[v + 1])] = np.arange(v + 1, n)
    return wtc.CSR(n + ALONE, m, rp, col), int((d.astype(np.int64) * (d - 1) // 2).sum())


def test_four_byte_offsets_up_to_their_end():
    t0 = time.perf_counter()

    def said(*what):
        print(f"{time.perf_counter() - t0:6.1f} s", *what, flush=True)

    g, W = _band((1 << 32) - 1)
    assert (1 << 32) - 64 < g.m < (1 << 32) - 1
    said("graph", g.n, g.m, W)
    ctx = wtc.Context(0)
    dg = ctx.upload(g, offset_bytes=4)
    del g
    gc.collect()
    said("uploaded")
    # the split count's top rows and dense part (the last 32,768 ranks) and,
    # with the vertices without edges alone on top, its list rows, up to the
    # end; then the other kernels
    for kernel, a in ((wtc.KERNEL_SPLIT, 32768), (wtc.KERNEL_SPLIT, 64), (wtc.KERNEL_ROWS, 0), (wtc.KERNEL_STAGED, 4096),
                      (wtc.KERNEL_WALK, 4096)):
        ctx.set_count_kernel(kernel)
        cnt, st = dg.count(8, a, stats=True)
        said("kernel", kernel, "a", a, st.as_dict())
        assert (cnt, st.wedges) == (W, W) and st.split == (kernel == wtc.KERNEL_SPLIT), (kernel, a)
        if kernel == wtc.KERNEL_SPLIT:  # the last wedges alone
            assert dg.count(8, a, W - 100000, W) == 100000
    dg.free()
    ctx.close()
