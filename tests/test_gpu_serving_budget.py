"""Serving under a memory budget that holds a graph's row count but not its
split count's workspace."""
import pytest

import wtc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mib,split", [(48, False), (512, True)])
def test_rmat18_with_and_without_room_for_the_workspace(gpu_ctx, mib, split):
    g = wtc.preprocess(wtc.gen_rmat(18, 16, seed=3))
    dg = gpu_ctx.upload(g)
    try:
        gpu_ctx.set_count_kernel(wtc.KERNEL_ROWS)
        expect = dg.count(8, 0)
    finally:
        gpu_ctx.set_count_kernel(wtc.KERNEL_WALK)
        dg.free()
    assert 1 << 27 <= g.wedges() < 1 << 28
    srv = wtc.Server(hbm_budget_bytes=mib << 20)
    try:
        gid = srv.register(g)
        rids = [srv.submit(gid, 8, 4096) for _ in range(3)]
        assert [srv.wait(r)[0] for r in rids] == [expect] * 3
        if split:  # no bitmap in HBM
            assert srv.wait(srv.submit(gid, 8, 32768))[0] == expect
        else:  # a bitmap of 128 MiB
            with pytest.raises(wtc.WtcError):
                srv.submit(gid, 8, 32768)
    finally:
        srv.close()
