"""The split count asked for no bitmap (a = 0): the row count and the staged
kernel up to 2^24 edges, the walk above."""
import pytest

import wtc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale,below", [(12, True), (20, True), (21, False)])
@pytest.mark.parametrize("ob", [4, 8])
def test_no_bitmap_whole_and_ranges(gpu_ctx, scale, below, ob):
    dg = wtc.DeviceGraph.gen_rmat(gpu_ctx, scale, 16, seed=5, offset_bytes=ob)
    try:
        assert (dg.m <= 1 << 24) == below
        gpu_ctx.set_count_kernel(wtc.KERNEL_STAGED)
        expect, st = dg.count(8, 0, stats=True)
        W = st.wedges
        gpu_ctx.set_count_kernel(wtc.KERNEL_SPLIT)
        cnt, st = dg.count(8, 0, stats=True)
        assert cnt == expect and st.split == 0 and st.wedges == W
        cuts = [0, W // 3, W // 3 + 1, W - W // 5, W]
        assert sum(dg.count(8, 0, lo, hi) for lo, hi in zip(cuts, cuts[1:])) == expect
    finally:
        dg.free()
        gpu_ctx.set_count_kernel(wtc.KERNEL_WALK)
