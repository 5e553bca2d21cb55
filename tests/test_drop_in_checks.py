"""The tc_GPU drop-ins on a CSR whose offsets do not fit its edge count: such a
call is refused from its two end offsets, before colInd, which may be shorter
than numEdges says, is read and before anything is allocated."""
import fake_gpu

PROGRAM = """
good = wtc.preprocess(wtc.gen_barabasi_albert(500, 3, seed=903))
rp, ci = good.row_ptr.copy(), good.col_ind.copy()
shifted = rp.copy()
shifted[0] = 1
assert wtc.tc_gpu_big(good, 5, 64) == 0  # the runtime stand-in works, and counts nothing
for wide in (False, True):
    for off, m in ((rp, good.m + 1), (rp, 2 * good.m), (rp, good.m - 1), (rp, 0xfffffff0), (shifted, good.m)):
        for arrays in (ci, ci[:0]):
            off_t = np.ascontiguousarray(off, dtype=np.uint64 if wide else np.uint32)
            col = arrays.ctypes.data_as(C.POINTER(C.c_uint32))
            cnt = C.c_uint64()
            fake.fake_reset()
            if wide:
                g = wtc._BigGraph(good.n, m, off_t.ctypes.data_as(C.POINTER(C.c_uint64)), col)
                rc = wtc._lib.wtc_tc_gpu_big(C.byref(g), 5, 64, None, C.byref(cnt))
            else:
                g = wtc._Graph32(good.n, m, off_t.ctypes.data_as(C.POINTER(C.c_uint32)), col)
                rc = wtc._lib.wtc_tc_gpu(C.byref(g), 5, 64, None, C.byref(cnt))
            case = (wide, m, int(off[0]))
            assert rc == -10, (case, rc)
            assert fake.fake_allocs() == 0 and fake.fake_copies() == 0, (case, fake.fake_allocs(), fake.fake_copies())
            assert fake.fake_launches() == 0, case
"""


def test_offsets_are_checked_before_anything_is_read_or_allocated(tmp_path):
    fake_gpu.run(tmp_path, PROGRAM)
