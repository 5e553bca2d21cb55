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


SMALL = BAND + """
graphs = [band(60 + i, 7) for i in range(4)]


def batches(ctx):
    b = wtc.Batch(ctx, graphs)
    yield launches(lambda: b.count([8] * 4, [0] * 4))
    yield launches(lambda: wtc.batch_count_host(ctx, graphs, [8] * 4, [0] * 4))


def serves(words, kernel):
    "Whether a served set of two graphs or more is counted by the kernel: no request alone is a set."
    srv = wtc.Server(hbm_budget_bytes=1 << 28, small_graph_words=words)
    gids = [srv.register(g) for g in graphs]
    seen = False
    for _ in range(300):
        def burst():
            sets = [srv.wait(r)[1].batch_graphs for r in [srv.submit(g, 8, 0) for g in gids * 16]]
            assert len(sets) == 64
        seen = seen or ran(launches(burst), kernel)
        if seen:
            break
    srv.close()
    return seen
"""


def test_small_graph_limit_is_kept_where_it_is_set(tmp_path):
    """Sets of small graphs go to the row count where it is the chosen kernel,
    but to the small-graph kernel where the caller has set its limit."""
    fake_gpu.run(tmp_path, SMALL + """
ctx = wtc.Context(0)
ctx.use_tuned(wtc.autotune_shape(graphs[0].n, graphs[0].m, graphs[0].wedges(), batch=True))
for limit, small in ((None, False), (20480, True), (0, False), (500, False), (40960, True)):
    if limit is not None:
        ctx.set_small_graphs(limit)
    for ks in batches(ctx):
        assert ran(ks, "k_count_small") == small and ran(ks, "k_rows") != small, (limit, ks)
# a batch kept by the program follows the setting, at the limit's own default, too
ctx = wtc.Context(0)
ctx.use_tuned(wtc.autotune_shape(graphs[0].n, graphs[0].m, graphs[0].wedges(), batch=True))
b = wtc.Batch(ctx, graphs)
assert ran(launches(lambda: b.count([8] * 4, [0] * 4)), "k_rows")
ctx.set_small_graphs(ctx.small_graphs()[0])
assert ran(launches(lambda: b.count([8] * 4, [0] * 4)), "k_count_small")
assert serves(20480, "k_count_small")
assert serves(0, "k_rows") and serves(-1, "k_rows")
""")
    fake_gpu.run(tmp_path, SMALL + """
ctx = wtc.Context(0)
ctx.use_tuned(wtc.autotune_shape(graphs[0].n, graphs[0].m, graphs[0].wedges(), batch=True))
assert all(ran(ks, "k_count_small") for ks in batches(ctx))
assert serves(0, "k_count_small")
""", {"WTC_SMALL_GRAPH_WORDS": "20480"})


def test_prefix_and_bitmap_of_a_count_that_has_none(tmp_path):
    """The debug copies of the wedge prefix and the bitmap are of the last count:
    after a row or split count, which leave neither, they are refused instead
    of showing an earlier count's."""
    fake_gpu.run(tmp_path, BAND + """
def refused(f):
    try:
        f()
    except wtc.WtcError as e:
        return e.code == -1
    return False


g = band(5000, 40)
ctx = wtc.Context(0)
dg = ctx.upload(g)
ctx.set_count_kernel(wtc.KERNEL_WALK)
dg.count(8, 64)
ctx.debug_prefix(g.n), ctx.debug_bitmap(128)
for kernel in (wtc.KERNEL_ROWS, wtc.KERNEL_SPLIT):
    ctx.set_count_kernel(kernel)
    dg.count(8, 64)
    assert refused(lambda: ctx.debug_prefix(g.n)) and refused(lambda: ctx.debug_bitmap(128)), kernel
    ctx.set_count_kernel(wtc.KERNEL_STAGED)
    dg.count(8, 64)
    ctx.debug_prefix(g.n), ctx.debug_bitmap(128)
""")


def test_small_sets_by_the_faster_kernel(tmp_path):
    """Where the row count is the chosen kernel it takes the sets of small graphs
    that it is the faster one for: small sets, graphs of few edges, or of many
    wedges an edge; large sets of sparse graphs of a thousand vertices or more go
    to the small-graph kernel."""
    fake_gpu.run(tmp_path, BAND + """
def sparse(n, m0):
    return wtc.preprocess(wtc.gen_barabasi_albert(n, m0, seed=3))


for g, k, small in ((sparse(64, 4), 2000, False), (sparse(250, 4), 2000, False), (sparse(1000, 4), 2000, True),
                    (sparse(1000, 4), 40, False), (sparse(1000, 16), 2000, False), (sparse(2000, 2), 2000, True),
                    (sparse(2000, 6), 2000, True), (sparse(2000, 6), 2, False), (sparse(4000, 2), 2000, True),
                    (band(130, 129), 500, False),
                    (sparse(4000, 8), 500, False)):  # the last has more words than the limit
    ctx = wtc.Context(0)
    ctx.use_tuned(wtc.autotune_shape(g.n, g.m, g.wedges(), batch=True))
    graphs = [g] * k
    b = wtc.Batch(ctx, graphs)
    for call in (lambda: b.count([8] * k, [0] * k), lambda: wtc.batch_count_host(ctx, graphs, [8] * k, [0] * k)):
        ks = launches(call)
        assert ran(ks, "k_count_small") == small and ran(ks, "k_rows") != small, (g.n, g.m, g.wedges(), k, ks)
""")


def test_graphs_without_wedges_take_no_tiles(tmp_path):
    """A set whose graphs have no wedges launches no counting kernel."""
    fake_gpu.run(tmp_path, BAND + """
ctx = wtc.Context(0)
ctx.set_count_kernel(wtc.KERNEL_ROWS)
star = wtc.preprocess(wtc.graph_from_pairs(np.stack([np.zeros(30000, int), 1 + np.arange(30000)], axis=1).astype(np.uint32)))
for graphs, kernel in (([star] * 3, False), ([star, band(20000, 5), star], True)):
    b = wtc.Batch(ctx, graphs)
    ks = launches(lambda: b.count([8] * 3, [0] * 3))
    assert ran(ks, "k_rows_init") and ran(ks, "k_rows") == kernel, ks
""")
