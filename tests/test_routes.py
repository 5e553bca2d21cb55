"""Which counting kernel the host code takes for a call, seen through a stand-in
HIP runtime: the rules that two entry points share give both the same kernel."""
import fake_gpu

BAND = """
def band(n, k):
    "Every vertex joined to the k after it."
    d = np.minimum(k, n - 1 - np.arange(n))
    rp = np.zeros(n + 1, dtype=np.uint64)
    np.cumsum(d, out=rp[1:])
    col = np.arange(int(rp[n])) - np.repeat(rp[:-1].astype(np.int64), d) + np.repeat(np.arange(n) + 1, d)
    return wtc.CSR(n, int(rp[n]), rp, col.astype(np.uint32))


def served(srv, gid, s, a):
    return srv.wait(srv.submit(gid, s, a))
"""


def test_large_graph_without_a_bitmap(tmp_path):
    """A whole graph counted with a = 0 where its size says split count: the row
    count, whatever its size, in a context as in the server; a range of it the
    walk."""
    fake_gpu.run(tmp_path, BAND + """
ctx = wtc.Context(0)
srv = wtc.Server(hbm_budget_bytes=1 << 30)
for n, k in ((20000, 420), (60000, 420)):  # 8.3 and 25 million edges
    g = band(n, k)
    t = wtc.autotune_shape(g.n, g.m, g.wedges())
    assert t.kernel == wtc.KERNEL_SPLIT, t.as_dict()
    ctx.use_tuned(t)
    dg = ctx.upload(g)
    gid = srv.register(g)
    for call in (lambda: dg.count(8, 0), lambda: served(srv, gid, 8, 0)):
        ks = launches(call)
        assert ran(ks, "k_rows") and not ran(ks, "k_walk"), (n, ks)
    for call in (lambda: dg.count(8, 4096), lambda: served(srv, gid, 8, 4096)):
        ks = launches(call)
        assert ran(ks, "k_split_rows"), (n, ks)
    ks = launches(lambda: dg.count(8, 0, 0, g.wedges() // 2))
    assert ran(ks, "k_walk") and not ran(ks, "k_rows"), (n, ks)
srv.close()
""")
