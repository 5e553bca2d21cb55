"""The tc_GPU drop-ins on a CSR whose offsets do not fit its edge count: such a
call is refused from its two end offsets, before colInd, which may be shorter
than numEdges says, is read and before anything is allocated."""
import os
import shutil
import subprocess

import pytest

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


THREADS = """
import resource
good = wtc.preprocess(wtc.gen_barabasi_albert(40000, 5, seed=903))  # rows for several threads
bad = wtc.CSR(good.n, good.m, good.row_ptr.copy(), good.col_ind.copy())
bad.col_ind[-1] = good.n
assert wtc.tc_gpu_big(good, 5, 64) == 0


def refused():
    try:
        wtc.tc_gpu_big(bad, 5, 64)
    except wtc.WtcError as e:
        return e.code == -10


# room for the call's buffers, not for another thread's stack; those that ended
# threads left behind are in use
import threading
ended = threading.Event()
for _ in range(16):
    threading.Thread(target=ended.wait, daemon=True).start()
now = int(open("/proc/self/statm").read().split()[0]) * resource.getpagesize()
resource.setrlimit(resource.RLIMIT_AS, (now + (3 << 20), -1))
try:
    threading.Thread(target=lambda: None).start()
    raise SystemExit("a thread could be started")
except RuntimeError:
    pass
assert wtc.tc_gpu_big(good, 5, 64) == 0
assert refused()
ended.set()
"""


@pytest.mark.parametrize("threads", [1, 4])
def test_without_a_thread_to_check_on(tmp_path, threads):
    """Where no thread can be started the check runs on the calling thread: no
    exception leaves the C entry, and none ends the process."""
    fake_gpu.run(tmp_path, THREADS, {"WTC_HOST_THREADS": str(threads)})


def test_the_check_lies_on_a_cache_line():
    """The check's loop is not inlined where its alignment, and with it a tc_GPU
    call's time, would change with other code."""
    if shutil.which("nm") is None:
        pytest.skip("needs nm")
    out = subprocess.run(["nm", "-C", os.path.join(fake_gpu.PKG, "libwtc.so")], check=True, capture_output=True, text=True)
    at = [int(x.split()[0], 16) for x in out.stdout.splitlines() if "int wtc::validate_oriented_rows_t<" in x]
    assert len(at) >= 2 and all(a % 64 == 0 for a in at), at
