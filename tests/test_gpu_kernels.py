"""Edge sizes of single kernels and dispatch rules, against the CPU oracle (bit-exact for
BFS, SSSP and CC)."""
import numpy as np
import pytest

from conftest import random_graph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 31, 255, 257, 65537, 262145, 524321])
def test_frontier_slices_cover_ragged_graphs(mg, oracle, device, n):
    # vertex counts around one slice, one workgroup and the 1024-workgroup share
    g = random_graph(mg, n, 6 * n, seed=n, symmetric=n % 2 == 1, wmax=16)
    src = int(np.argmax(g.degrees()))
    srcs = [src, n - 1, 0]
    with mg.Graph(g, symmetric=n % 2 == 1) as dg:
        assert np.array_equal(dg.bfs(src), oracle.bfs(g.row_offsets, g.col_idx, src))
        assert np.array_equal(dg.sssp(src), oracle.sssp(g.row_offsets, g.col_idx, g.values, src))
        for got, s in zip(dg.bfs_batch(srcs), srcs):
            assert np.array_equal(got, oracle.bfs(g.row_offsets, g.col_idx, s))
        for got, s in zip(dg.sssp_batch(srcs), srcs):
            assert np.array_equal(got, oracle.sssp(g.row_offsets, g.col_idx, g.values, s))


# ---------------------------------------------------------------- teams (narrow levels)
def _chain(mg, lengths, hubs, seed, symmetric=True):
    """Chains of the given lengths joined by stars: hubs[i] leaves around the end of chain i."""
    src, dst, v = [], [], 0
    for ln, hub in zip(lengths, hubs):
        ids = np.arange(v, v + ln)
        src.append(ids[:-1]), dst.append(ids[1:])
        end = v + ln - 1
        v += ln
        if hub:
            leaves = np.arange(v, v + hub)
            src.append(np.full(hub, end)), dst.append(leaves)
            v += hub
            src.append(leaves[-1:]), dst.append([v])  # the next chain starts behind the last leaf
    src, dst = np.concatenate(src).astype(np.int32), np.concatenate(dst).astype(np.int32)
    keep = dst < v
    flags = mg.MG_CSR_SORT_COLS | mg.MG_CSR_DEDUPE | (mg.MG_CSR_SYMMETRIZE if symmetric else 0)
    g = mg.csr_from_edges(v, src[keep], dst[keep], flags)
    g.values = mg.hash_weights(g, seed, 9)
    return g


def _team_graph(mg, which):
    if which == "path":
        return _chain(mg, [2500], [0], 3), True
    if which == "hubs":  # stars around the record, member and vertex limits of a team
        return _chain(mg, [40, 30, 30, 30, 20], [5, 1020, 1021, 9000, 0], 4), True
    if which == "directed":  # sinks all along
        return _chain(mg, [60, 200, 30], [33, 700, 0], 5, symmetric=False), False
    if which == "zero":
        g = mg.grid_graph(97, 61, seed=8, weight_max=3)
        g.values = g.values - 1
        return g, True
    if which == "tails":  # chains into a dense graph and out of it
        r = mg.rmat_graph(12, 16, seed=4)
        k, n, hub = 60, r.n, int(np.argmax(r.degrees()))
        a, b = np.arange(n, n + k), np.arange(n + k, n + 2 * k)
        src = np.concatenate([np.repeat(np.arange(n), np.diff(r.row_offsets)), a[:-1], b[:-1], [a[-1], hub]])
        dst = np.concatenate([r.col_idx, a[1:], b[1:], [hub, b[0]]])
        g = mg.csr_from_edges(n + 2 * k, src.astype(np.int32), dst.astype(np.int32),
                              mg.MG_CSR_SYMMETRIZE | mg.MG_CSR_DEDUPE | mg.MG_CSR_SORT_COLS)
        g.values = mg.hash_weights(g, 3, 64)
        return g, True
    w, h = which
    return mg.grid_graph(w, h, seed=w, weight_max=16), True


@pytest.mark.parametrize("which", ["path", "hubs", "directed", "zero", "tails", (64, 64), (701, 13), (399, 403)])
def test_teams_match_the_oracle(mg, oracle, device, which):
    g, sym = _team_graph(mg, which)
    with mg.Graph(g, symmetric=sym) as dg:
        for src in {0, g.n // 2, g.n - 1}:
            d, st = dg.bfs(src, stats=True)
            exp = oracle.bfs(g.row_offsets, g.col_idx, src)
            assert np.array_equal(d, exp)
            assert st.edges_traversed == oracle.teps_edges(g.row_offsets, exp)
            exp = oracle.sssp(g.row_offsets, g.col_idx, g.values, src)
            for delta in (0, 1, 7, -1):
                assert np.array_equal(dg.sssp(src, mg.options(sssp_delta=delta)), exp), (src, delta)


@pytest.mark.parametrize("limit", [8, 9, 10, 11, 40])
def test_team_stops_at_the_level_limit(mg, oracle, device, limit):
    g = mg.grid_graph(90, 70, seed=2, weight_max=16)
    with mg.Graph(g, symmetric=True) as dg:
        d, st = dg.bfs(0, mg.options(iter_num=limit), stats=True)
    exp = oracle.bfs(g.row_offsets, g.col_idx, 0)
    assert st.iterations == limit
    assert np.array_equal(d, np.where((exp >= 0) & (exp <= limit), exp, -1))


def test_teams_of_several_graphs_at_once(mg, oracle, device):
    """Teams on several streams share the GPU; none waits for a workgroup that is not running."""
    import threading

    hosts = [mg.grid_graph(150 + 31 * i, 120, seed=i, weight_max=16) for i in range(6)]
    graphs = [mg.Graph(h, symmetric=True) for h in hosts]
    got = [None] * len(hosts)

    def work(i):
        got[i] = [(graphs[i].bfs(s), graphs[i].sssp(s)) for s in (0, 77, 5000)]

    ts = [threading.Thread(target=work, args=(i,)) for i in range(len(hosts))]
    [t.start() for t in ts]
    [t.join() for t in ts]
    for h, rows in zip(hosts, got):
        for s, (b, d) in zip((0, 77, 5000), rows):
            assert np.array_equal(b, oracle.bfs(h.row_offsets, h.col_idx, s))
            assert np.array_equal(d, oracle.sssp(h.row_offsets, h.col_idx, h.values, s))
    [g.close() for g in graphs]


# ---------------------------------------------------------------- batched BFS by levels
def _clique_chain(mg, cliques, size, symmetric=True):
    """A chain of cliques: diameter about `cliques`, mean degree above 8."""
    src, dst = [], []
    for c in range(cliques):
        ids = np.arange(c * size, (c + 1) * size)
        a, b = np.meshgrid(ids, ids)
        src.append(a.ravel()), dst.append(b.ravel())
        if c + 1 < cliques:
            src.append([ids[-1]]), dst.append([ids[-1] + 1])
    flags = mg.MG_CSR_DROP_LOOPS | mg.MG_CSR_SORT_COLS | mg.MG_CSR_DEDUPE | (mg.MG_CSR_SYMMETRIZE if symmetric else 0)
    return mg.csr_from_edges(cliques * size, np.concatenate(src).astype(np.int32), np.concatenate(dst).astype(np.int32),
                             flags)


@pytest.mark.parametrize("cliques", [3, 5, 9, 15, 16, 17, 40])
@pytest.mark.parametrize("symmetric,k", [(True, 5), (False, 70)])
def test_batch_levels_at_their_limits(mg, oracle, device, cliques, symmetric, k):
    # two levels a clique: depths around the 8, 16 and 32 levels kept, and searches too deep for them
    g = _clique_chain(mg, cliques, 40, symmetric)
    srcs = np.random.default_rng(k).integers(0, g.n, k).astype(np.int32)
    srcs[:2] = [0, g.n - 1]
    exp = np.stack([oracle.bfs(g.row_offsets, g.col_idx, int(s)) for s in srcs])
    for relabel in (False, True):
        with mg.Graph(g, symmetric=symmetric, build_csc=not symmetric, relabel=relabel) as dg:
            for alpha in (0, 1, 1 << 20):  # the default switch, push only, pull early
                got, st = dg.bfs_batch(srcs, mg.options(batch_alpha=alpha), stats=True)
                assert np.array_equal(got, exp)
                assert st.edges_traversed == sum(oracle.teps_edges(g.row_offsets, r) for r in exp)
                assert st.vertices_reached == int((exp >= 0).sum())
            limit = 2 + cliques // 3
            got = dg.bfs_batch(srcs, mg.options(iter_num=limit))
            assert np.array_equal(got, np.where(exp <= limit, exp, -1))


def test_batch_levels_long_in_lists(mg, oracle, device):
    # hubs on both sides of the pieces a pull cuts long in-lists into
    rng = np.random.default_rng(5)
    n, hubs = 12000, [33, 1056, 1057, 2081, 9000]
    src, dst = [rng.integers(0, n, 6 * n)], [rng.integers(0, n, 6 * n)]
    for i, d in enumerate(hubs):
        src.append(np.full(d, i)), dst.append(rng.choice(np.arange(10, n), d, replace=False))
    g = mg.csr_from_edges(n, np.concatenate(src).astype(np.int32), np.concatenate(dst).astype(np.int32),
                          mg.MG_CSR_SYMMETRIZE | mg.MG_CSR_DROP_LOOPS | mg.MG_CSR_DEDUPE | mg.MG_CSR_SORT_COLS)
    srcs = rng.integers(0, n, 256).astype(np.int32)
    with mg.Graph(g, symmetric=True) as dg:
        rows = dg.bfs_batch(srcs, mg.options(batch_alpha=1 << 20))
    for j in range(0, 256, 15):
        assert np.array_equal(rows[j], oracle.bfs(g.row_offsets, g.col_idx, int(srcs[j])))


# ---------------------------------------------------------------- batched searches by teams
@pytest.mark.parametrize("which", ["path", "directed", "zero", (33, 31), (260, 19), "random"])
@pytest.mark.parametrize("k", [1, 9, 256])
def test_batch_teams_match_the_oracle(mg, oracle, device, which, k):
    # sparse graphs; "random" outgrows the teams' queues and falls back to the shared batch
    if which == "random":
        g, sym = random_graph(mg, 120000, 350000, 3, wmax=20), True
    elif which == "path":
        g, sym = _chain(mg, [300], [0], 3), True
    else:
        g, sym = _team_graph(mg, which)
    assert g.m < 8 * g.n
    rng = np.random.default_rng(k)
    srcs = rng.integers(0, g.n, k).astype(np.int32)
    pick = sorted({0, k // 2, k - 1})
    for relabel in (False, True):
        with mg.Graph(g, symmetric=sym, relabel=relabel) as dg:
            for _ in range(2):
                rows, st = dg.bfs_batch(srcs, stats=True)
                assert st.vertices_reached == int((rows >= 0).sum())
                assert st.edges_traversed == sum(oracle.teps_edges(g.row_offsets, r) for r in rows)
                srows = dg.sssp_batch(srcs)
                for j in pick:
                    assert np.array_equal(rows[j], oracle.bfs(g.row_offsets, g.col_idx, int(srcs[j])))
                    exp = oracle.sssp(g.row_offsets, g.col_idx, g.values, int(srcs[j]))
                    assert np.array_equal(srows[j], exp)
            for delta in (1, 5, -1):
                assert np.array_equal(dg.sssp_batch(srcs[:3], mg.options(sssp_delta=delta)), srows[:3])
            # stopped short, then whole again: the teams' bitmaps are clean
            cut = dg.bfs_batch(srcs, mg.options(iter_num=3))
            assert np.array_equal(cut, np.where(rows <= 3, rows, -1))
            dg.sssp_batch(srcs, mg.options(iter_num=3))
            assert np.array_equal(dg.bfs_batch(srcs), rows) and np.array_equal(dg.sssp_batch(srcs), srows)


def test_batch_teams_source_sets(mg, oracle, device):
    g = mg.grid_graph(70, 45, seed=3, weight_max=9)
    rng = np.random.default_rng(2)
    row_of = np.concatenate([np.arange(5), rng.integers(0, 5, 200)]).astype(np.int32)
    srcs = rng.integers(0, g.n, 205).astype(np.int32)
    srcs[7] = srcs[8] = srcs[row_of.tolist().index(row_of[7])]  # repeated sources
    with mg.Graph(g, symmetric=True) as dg:
        rows, srows = dg.bfs_batch_sets(row_of, srcs, 5), dg.sssp_batch_sets(row_of, srcs, 5)
    for r in range(5):
        mine = [int(s) for s in srcs[row_of == r]]
        b = np.stack([oracle.bfs(g.row_offsets, g.col_idx, s) for s in mine]).astype(np.int64)
        assert np.array_equal(rows[r], np.where((b < 0).all(0), -1, np.where(b < 0, 1 << 40, b).min(0)))
        d = np.stack([oracle.sssp(g.row_offsets, g.col_idx, g.values, s) for s in mine])
        assert np.array_equal(srows[r], d.min(0))


# ---------------------------------------------------------------- batched SSSP by pulling
@pytest.mark.parametrize("k", [1, 3, 32, 33, 64, 65, 128, 129, 256])
@pytest.mark.parametrize("symmetric", [True, False])
def test_batch_pull_row_widths(mg, oracle, device, k, symmetric):
    # row widths around every group size; hubs around the piece length; a small component
    rng = np.random.default_rng(k)
    n, hubs = 3000, [511, 512, 513, 1024, 1025, 2500]
    src, dst = [rng.integers(0, n - 20, 8 * n)], [rng.integers(0, n - 20, 8 * n)]
    for i, d in enumerate(hubs):
        a, b = np.full(d, i), rng.choice(np.arange(10, n - 20), d, replace=False)
        src += [a, b]
        dst += [b, a]
    src.append(np.arange(n - 10, n - 1)), dst.append(np.arange(n - 9, n))
    flags = mg.MG_CSR_DROP_LOOPS | mg.MG_CSR_DEDUPE | mg.MG_CSR_SORT_COLS | (mg.MG_CSR_SYMMETRIZE if symmetric else 0)
    g = mg.csr_from_edges(n, np.concatenate(src).astype(np.int32), np.concatenate(dst).astype(np.int32), flags)
    g.values = mg.hash_weights(g, k, 50) - 1
    assert g.m >= 8 * g.n
    srcs = rng.integers(0, n, k).astype(np.int32)
    srcs[0] = n - 10  # in the small component
    exp = np.stack([oracle.sssp(g.row_offsets, g.col_idx, g.values, int(s)) for s in srcs])
    for relabel in (False, True):
        with mg.Graph(g, symmetric=symmetric, build_csc=not symmetric, relabel=relabel) as dg:
            for _ in range(2):
                got, st = dg.sssp_batch(srcs, stats=True)
                assert np.array_equal(got, exp)
            assert st.vertices_reached == int((exp != 2**31 - 1).sum())
            assert st.edges_traversed == sum(oracle.teps_edges(g.row_offsets, r, 2**31 - 1) for r in exp)
            assert np.array_equal(dg.sssp_batch(srcs[:1])[0], exp[0])  # another width on the same state


@pytest.mark.parametrize("cliques", [20, 47, 48, 60])
def test_batch_pull_falls_back_when_deep(mg, oracle, device, cliques):
    g = _clique_chain(mg, cliques, 20)
    g.values = mg.hash_weights(g, 2, 30)
    srcs = np.array([0, g.n // 2, g.n - 1], np.int32)
    with mg.Graph(g, symmetric=True) as dg:
        for _ in range(2):
            for got, s in zip(dg.sssp_batch(srcs), srcs):
                assert np.array_equal(got, oracle.sssp(g.row_offsets, g.col_idx, g.values, int(s)))


def test_batch_pull_huge_weights(mg, oracle, device):
    # distances at the top of the 32-bit range: sums past INT_MAX never improve anything
    g = random_graph(mg, 400, 3000, 3, wmax=7)
    g.values = (g.values * 150_000_000).astype(np.int32)
    srcs = np.arange(5, dtype=np.int32)
    with mg.Graph(g, symmetric=True) as dg:
        for got, s in zip(dg.sssp_batch(srcs), srcs):
            assert np.array_equal(got, dg.sssp(int(s)))


# ---------------------------------------------------------------- PageRank
@pytest.mark.parametrize("relabel", [False, True])
@pytest.mark.parametrize("hubs", [True, False])
@pytest.mark.parametrize("n", [3100, 15359, 15360, 15361, 40003])
def test_pagerank_list_lengths(mg, oracle, device, n, hubs, relabel):
    # in-degrees around a lane's, a wave's and a piece's edges, first, last and between low ones;
    # sources all over the ids or, for a graph without hubs in LDS, past the ids kept there
    rng = np.random.default_rng(n + hubs)
    degs = [1, 2, 47, 48, 49, 63, 64, 65, 0, 255, 256, 257, 511, 512, 513, 1024, 1025, 3000]
    at = [0, 1, 2, *sorted(rng.choice(np.arange(3, n - 3), len(degs) - 6, replace=False)), n - 3, n - 2, n - 1]
    low = rng.integers(0, 5, n)
    low[at] = rng.permutation(degs)
    far = not hubs and n > 2 * 15360
    src = np.concatenate([rng.choice(np.arange(15360 if far else 0, n), d, replace=False) for d in low])
    g = mg.csr_from_edges(n, src.astype(np.int32), np.repeat(np.arange(n), low).astype(np.int32), mg.MG_CSR_SORT_COLS)
    # all terms are positive: a list's sum errs by at most 48 (a lane), or 32 + 6 + 12 (pieces), roundings,
    # the rank by 4 more, and 0.85 of an iteration's relative error goes into the next
    rtol = (50 + 4) * 2.0**-24 / 0.15
    with mg.Graph(g, build_csc=True, relabel=relabel) as dg:
        for iters, tol in ((1, 0.0), (12, 0.0), (12, 1e-9)):
            exp, _, _ = oracle.pr_jacobi_f64(g.row_offsets, g.col_idx, iters=iters)
            for _ in range(2):
                got, st = dg.pagerank(mg.options(pr_mode=mg.MG_PR_ALL, iter_num=iters, pr_tol=tol), stats=True)
                assert st.iterations == iters
                assert np.max(np.abs(got - exp) / exp) <= rtol
        got, st = dg.pagerank(stats=True)
    exp, it = oracle.pr_gas(g.row_offsets, g.col_idx)
    assert abs(st.iterations - it) <= 1
    assert np.max(np.abs(got.astype(np.float64) - exp)) / n <= 1e-6


# ---------------------------------------------------------------- personalized PageRank
@pytest.mark.parametrize("relabel", [False, True])
@pytest.mark.parametrize("n", [1500, 1537, 4096])
def test_ppr_list_lengths(mg, oracle, device, n, relabel):
    # in-degrees around a block's, a team's and a piece's edges; empty lists first and last
    rng = np.random.default_rng(n)
    low = rng.integers(0, 12, n)
    degs = [7, 8, 9, 15, 16, 17, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513, 1400]
    low[rng.choice(np.arange(2, n - 2), len(degs), replace=False)] = degs
    low[[0, 1, n - 2, n - 1]] = [0, 1, 3, 0]
    src = np.concatenate([rng.choice(n, d, replace=False) for d in low])
    g = mg.csr_from_edges(n, src.astype(np.int32), np.repeat(np.arange(n), low).astype(np.int32), mg.MG_CSR_SORT_COLS)
    srcs = rng.integers(0, n, 64).astype(np.int32)
    # all terms are positive: a list's sum errs by at most 3 + 4 + 3 + 6 roundings (block, partial sum, their
    # tree, pieces), the rank by 4 more, and 0.85 of an iteration's relative error goes into the next
    rtol = 20 * 2.0**-24 / 0.15
    with mg.Graph(g, build_csc=True, relabel=relabel) as dg:
        for iters in (1, 2, 3, 20):
            o = mg.options(ppr_iters=iters)
            full = dg.ppr_batch(srcs, o)
            for j in (0, 40, 63):
                exp = oracle.ppr(g.row_offsets, g.col_idx, int(srcs[j]), iters=iters)
                assert np.all(np.abs(full[j] - exp) <= rtol * exp + 1e-37)
            for k in (1, 8, 9, 16, 17, 32, 33):  # the other row widths
                assert np.array_equal(dg.ppr_batch(srcs[:k], o).view(np.int32), full[:k].view(np.int32))


def test_ppr_rows_past_4_gib(mg, oracle, device):
    # 64 columns of 2^24 + 3 vertices: the widest rows' offsets need more than 32 bits
    n = (1 << 24) + 3
    rng = np.random.default_rng(4)
    src, dst = rng.integers(0, n, 2 * n, dtype=np.int32), rng.integers(0, n, 2 * n, dtype=np.int32)
    hub = rng.integers(n - 50, n, 4000, dtype=np.int32)
    src, dst = np.concatenate([src, hub]), np.concatenate([dst, np.full(4000, n - 1, np.int32)])
    g = mg.csr_from_edges(n, src, dst, mg.MG_CSR_SORT_COLS)
    srcs = np.concatenate([np.arange(n - 30, n), rng.integers(0, n, 3)]).astype(np.int32)
    o = mg.options(ppr_iters=2)
    with mg.Graph(g, build_csc=True) as dg:
        few = dg.ppr_batch(srcs[:8], o)  # rows of 8 columns: below 4 GiB
        full = dg.ppr_batch(srcs, o)
    assert np.array_equal(full[:8].view(np.int32), few.view(np.int32))
    for j in (0, 29, 32):
        assert np.max(np.abs(full[j] - oracle.ppr(g.row_offsets, g.col_idx, int(srcs[j]), iters=2))) <= 1e-6


@pytest.mark.parametrize("edges", [0, 1, 2, 3, 4, 5, 9])
def test_ppr_tiny_adjacency(mg, oracle, device, edges):
    # fewer edges than the loads of a block are wide
    src, dst = np.arange(edges, dtype=np.int32), np.arange(1, edges + 1, dtype=np.int32)
    g = mg.csr_from_edges(edges + 2, src, dst, 0)
    with mg.Graph(g, build_csc=True) as dg:
        for s, got in enumerate(dg.ppr_batch(np.arange(min(edges + 2, 8), dtype=np.int32))):
            assert np.max(np.abs(got - oracle.ppr(g.row_offsets, g.col_idx, s))) <= 1e-6


# ---------------------------------------------------------------- what follows a search
@pytest.mark.parametrize("relabel", [False, True])
@pytest.mark.parametrize("n", [1, 3, 1023, 1025, 262144, 262145, 1100003])
def test_results_reach_every_kind_of_output(mg, oracle, device, n, relabel):
    # vertex counts around the workgroups of the closing kernel and the host copies made ahead
    import ctypes as C

    hip = C.CDLL("libamdhip64.so")
    dev, pin = C.c_void_p(), C.c_void_p()
    assert hip.hipMalloc(C.byref(dev), C.c_size_t(4 * n + 8)) == 0
    assert hip.hipHostMalloc(C.byref(pin), C.c_size_t(4 * n), 0) == 0
    g = random_graph(mg, n, 3 * n, seed=n, symmetric=True, wmax=9)
    srcs = [int(np.argmax(g.degrees())), 0, n - 1]  # searches of other lengths than the last one's
    with mg.Graph(g, symmetric=True, relabel=relabel) as dg:
        def outputs(name, *args):
            fn, st = getattr(mg.lib(), name), mg.Stats()

            def call(ptr, on_device, stats):
                o = mg.options(out_on_device=on_device, pr_mode=mg.MG_PR_ALL, iter_num=5 if name == "mg_pagerank" else 100000)
                mg.check(fn(dg.handle, *args, C.c_void_p(ptr), C.byref(o), C.byref(st) if stats else None))

            host, bare, raw = np.empty(n, np.int32), np.empty(n, np.int32), np.empty(4 * n + 8, np.uint8)
            call(host.ctypes.data, 0, True)
            call(bare.ctypes.data, 0, False)
            call(pin.value, 0, True)
            assert np.array_equal(bare, host)
            assert np.array_equal(np.ctypeslib.as_array(C.cast(pin, C.POINTER(C.c_int32)), (n,)), host)
            for at, stats in ((4, True), (4, False), (1, True)):  # (odd addresses too)
                raw[:] = 0xA5
                assert hip.hipMemcpy(dev, raw.ctypes.data_as(C.c_void_p), C.c_size_t(raw.nbytes), 1) == 0
                call(dev.value + at, 1, stats)
                assert hip.hipMemcpy(raw.ctypes.data_as(C.c_void_p), dev, C.c_size_t(raw.nbytes), 2) == 0
                assert np.array_equal(raw[at:at + 4 * n].copy().view(np.int32), host)
                assert np.all(raw[:at] == 0xA5) and np.all(raw[at + 4 * n:] == 0xA5)
            call(None, 0, True)
            return host, st

        for src in srcs:
            d, st = outputs("mg_bfs", src)
            assert np.array_equal(d, oracle.bfs(g.row_offsets, g.col_idx, src))
            assert st.vertices_reached == int((d >= 0).sum())
            assert st.edges_traversed == oracle.teps_edges(g.row_offsets, d)
            d, st = outputs("mg_sssp", src)
            assert np.array_equal(d, oracle.sssp(g.row_offsets, g.col_idx, g.values, src))
            assert st.edges_traversed == oracle.teps_edges(g.row_offsets, d, 2**31 - 1)
        d, st = outputs("mg_cc")
        assert np.array_equal(d, oracle.cc(g.row_offsets, g.col_idx))
        assert (st.vertices_reached, st.edges_traversed) == (n, g.m)
        outputs("mg_pagerank")
    hip.hipFree(dev)
    hip.hipHostFree(pin)


# ---------------------------------------------------------------- connected components
@pytest.mark.parametrize("sort", [False, True])
@pytest.mark.parametrize("n,parts", [(40, 1), (257, 3), (5000, 7), (70001, 2), (300007, 40)])
def test_cc_dense_components(mg, oracle, device, n, parts, sort):
    # mean degree above 8; first neighbours above and below their vertex, lists of any order, hubs
    # and isolated vertices outside the sampled component
    rng = np.random.default_rng(n + sort)
    part = rng.integers(0, parts, n)
    ids = [np.flatnonzero(part == k) for k in range(parts)]
    src = np.concatenate([rng.choice(i[: max(1, len(i) * 3 // 4)], 8 * len(i)) for i in ids if len(i)])
    dst = np.concatenate([rng.choice(i[: max(1, len(i) * 3 // 4)], 8 * len(i)) for i in ids if len(i)])
    small = min(ids, key=len)
    src, dst = np.concatenate([src, np.full(len(small), small[0])]), np.concatenate([dst, small])  # a hub
    flags = mg.MG_CSR_SYMMETRIZE | mg.MG_CSR_DROP_LOOPS | (mg.MG_CSR_SORT_COLS | mg.MG_CSR_DEDUPE if sort else 0)
    g = mg.csr_from_edges(n, src.astype(np.int32), dst.astype(np.int32), flags)
    assert g.m >= 8 * n
    exp = oracle.cc(g.row_offsets, g.col_idx)
    with mg.Graph(g, symmetric=True) as dg:
        for _ in range(2):
            got, st = dg.cc(stats=True)
            assert np.array_equal(got, exp)
            assert (st.vertices_reached, st.edges_traversed, st.iterations) == (n, g.m, 1)


# ---------------------------------------------------------------- SSSP pull and wide push tasks
@pytest.mark.parametrize("symmetric", [False, True])
@pytest.mark.parametrize("n", [2000, 2049, 300001])
def test_sssp_dense_task_sizes(mg, oracle, device, n, symmetric):
    # in-lists around the pieces and ranges of the smallest tasks; at the last size (over 5M edges)
    # around those of larger ones
    rng = np.random.default_rng(n)
    big = n > 10**5
    low = rng.integers(0, 40 if big else 16, n)
    t = 704 if big else 512  # edges a task (directed)
    degs = [t // 4 - 1, t // 4, t // 4 + 1, t - 1, t, t + 1, 2 * t, 2 * t + 1]
    low[[0, 1, n - 1, *rng.choice(np.arange(40, n - 40), 5, replace=False)]] = degs
    low[64:96] = t // 4  # a word of the longest lists that are not cut
    dst = np.repeat(np.arange(n), low).astype(np.int32)
    src = rng.integers(0, n, len(dst)).astype(np.int32)
    flags = mg.MG_CSR_SORT_COLS | (mg.MG_CSR_SYMMETRIZE if symmetric else 0)
    g = mg.csr_from_edges(n, src, dst, flags)
    g.values = mg.hash_weights(g, 5, 64) - 1
    with mg.Graph(g, symmetric=symmetric, build_csc=not symmetric) as dg:
        pulls = 0
        for s in (int(np.argmax(g.degrees())), 70, n - 1):
            got, st = dg.sssp(s, stats=True)
            assert np.array_equal(got, oracle.sssp(g.row_offsets, g.col_idx, g.values, s))
            pulls += st.bottom_up_levels
        assert pulls or not big


@pytest.mark.parametrize("k", [100, 256])
@pytest.mark.parametrize("depth", [10, 12, 13, 15])
def test_batch_teams_grow(mg, oracle, device, depth, k):
    # binary trees whose levels outgrow teams of 2, 4 and 8 workgroups, and the largest
    n = 2 ** (depth + 1) - 1
    v = np.arange(1, n)
    g = mg.csr_from_edges(n, ((v - 1) // 2).astype(np.int32), v.astype(np.int32), mg.MG_CSR_SYMMETRIZE | mg.MG_CSR_SORT_COLS)
    g.values = mg.hash_weights(g, depth, 9)
    srcs = np.random.default_rng(depth).integers(0, n, k).astype(np.int32)
    srcs[:3] = [0, n - 1, n // 2]
    bfs = np.stack([oracle.bfs(g.row_offsets, g.col_idx, int(s)) for s in srcs])
    sssp = np.stack([oracle.sssp(g.row_offsets, g.col_idx, g.values, int(s)) for s in srcs])
    with mg.Graph(g, symmetric=True) as dg:
        for _ in range(2):
            got, st = dg.bfs_batch(srcs, stats=True)
            assert np.array_equal(got, bfs)
            assert st.vertices_reached == k * n and st.edges_traversed == k * g.m
            got, st = dg.sssp_batch(srcs, stats=True)
            assert np.array_equal(got, sssp)
            assert st.vertices_reached == k * n
        assert np.array_equal(dg.bfs_batch(srcs[:5]), bfs[:5])


def test_batch_pull_falls_back_whatever_the_bucket_width(mg, oracle, device):
    # the pushed route's steps beside the pulled route's, at a width that once named both
    g = _clique_chain(mg, 60, 20)
    g.values = mg.hash_weights(g, 2, 30)
    srcs = np.array([0, g.n // 2, g.n - 1], np.int32)
    with mg.Graph(g, symmetric=True) as dg:
        for got, s in zip(dg.sssp_batch(srcs, mg.options(sssp_delta=0x9011 + len(srcs))), srcs):
            assert np.array_equal(got, oracle.sssp(g.row_offsets, g.col_idx, g.values, int(s)))


# ---------------------------------------------------------------- where batched results go
@pytest.mark.parametrize("relabel", [False, True])
@pytest.mark.parametrize("which", ["sparse", "dense", "wide"])
def test_batched_results_reach_every_kind_of_output(mg, oracle, device, which, relabel):
    # the routes by teams, by levels and by pulling, and the general one: device memory at even and odd
    # addresses, fine-grained device memory, managed and pinned memory named as device pointers, host memory
    import ctypes as C

    if which == "sparse":
        g = mg.grid_graph(61, 37, seed=5, weight_max=9)
    elif which == "dense":
        g = random_graph(mg, 1501, 12000, 6, wmax=30)
    else:
        g = random_graph(mg, 120000, 350000, 3, wmax=20)
    k, n = 3, g.n
    srcs = np.array([0, n // 2, n - 1], np.int32)
    size, I32P = 4 * k * n, C.POINTER(C.c_int32)
    hip = C.CDLL("libamdhip64.so")
    kinds = {"device": lambda p: hip.hipMalloc(p, C.c_size_t(size + 8)),
             "fine-grained": lambda p: hip.hipExtMallocWithFlags(p, C.c_size_t(size + 8), C.c_uint(1)),
             "managed": lambda p: hip.hipMallocManaged(p, C.c_size_t(size + 8), C.c_uint(1)),
             "pinned": lambda p: hip.hipHostMalloc(p, C.c_size_t(size + 8), C.c_uint(0))}
    mem = {}
    for kind, alloc in kinds.items():
        mem[kind] = C.c_void_p()
        assert alloc(C.byref(mem[kind])) == 0
    with mg.Graph(g, symmetric=True, relabel=relabel) as dg:
        for name, one in (("mg_bfs_batch", lambda s: oracle.bfs(g.row_offsets, g.col_idx, s)),
                          ("mg_sssp_batch", lambda s: oracle.sssp(g.row_offsets, g.col_idx, g.values, s))):
            exp = np.stack([one(int(s)) for s in srcs])
            raw = np.empty(size + 8, np.uint8)

            def call(ptr, on_device):
                o, st = mg.options(out_on_device=on_device), mg.Stats()
                mg.check(getattr(mg.lib(), name)(dg.handle, srcs.ctypes.data_as(I32P), k, C.c_void_p(ptr), C.byref(o),
                                                 C.byref(st)))
                assert st.vertices_reached == int(((exp >= 0) & (exp != 2**31 - 1)).sum())

            host = np.zeros((k, n), np.int32)
            call(host.ctypes.data, 0)
            assert np.array_equal(host, exp)
            for kind, p in mem.items():
                for at in (0, 4, 1):
                    raw[:] = 0xA5
                    assert hip.hipMemcpy(p, raw.ctypes.data_as(C.c_void_p), C.c_size_t(raw.nbytes), 4) == 0
                    call(p.value + at, 1)
                    assert hip.hipMemcpy(raw.ctypes.data_as(C.c_void_p), p, C.c_size_t(raw.nbytes), 4) == 0
                    assert np.array_equal(raw[at:at + size].copy().view(np.int32).reshape(k, n), exp), (name, kind, at)
                    assert np.all(raw[:at] == 0xA5) and np.all(raw[at + size:] == 0xA5), (name, kind, at)
            call(None, 0)
            call(None, 1)
    for kind, p in mem.items():
        (hip.hipHostFree if kind == "pinned" else hip.hipFree)(p)


@pytest.mark.parametrize("which", ["teams", "levels", "pull"])
@pytest.mark.parametrize("kth", [1, 2, 3, 4, 5, 6, 7, 8])
def test_batched_routes_refused_memory_go_the_general_way(mg, oracle, device, monkeypatch, which, kth):
    # the kth allocation of a call is refused: one that only a faster route needs fails no call
    import ctypes as C

    g = mg.grid_graph(61, 37, seed=5, weight_max=9) if which == "teams" else random_graph(mg, 1501, 12000, 6, wmax=30)
    srcs = np.array([0, g.n // 2, g.n - 1], np.int32)
    bfs = np.stack([oracle.bfs(g.row_offsets, g.col_idx, int(s)) for s in srcs])
    sssp = np.stack([oracle.sssp(g.row_offsets, g.col_idx, g.values, int(s)) for s in srcs])
    with mg.Graph(g, symmetric=True) as dg:
        if which == "levels":  # the context, which both routes need, without the rows of a host result
            hip, p, o = C.CDLL("libamdhip64.so"), C.c_void_p(), mg.options(out_on_device=1)
            assert hip.hipMalloc(C.byref(p), C.c_size_t(12 * g.n)) == 0
            mg.check(mg.lib().mg_bfs_batch(dg.handle, srcs.ctypes.data_as(C.POINTER(C.c_int32)), 3, p, C.byref(o), None))
            hip.hipFree(p)
        monkeypatch.setenv("MG_FAIL_ALLOC_AT", str(kth))
        rows = dg.sssp_batch(srcs) if which == "pull" else dg.bfs_batch(srcs)
        monkeypatch.delenv("MG_FAIL_ALLOC_AT")
        assert np.array_equal(rows, sssp if which == "pull" else bfs)
        for _ in range(2):
            assert np.array_equal(dg.bfs_batch(srcs), bfs) and np.array_equal(dg.sssp_batch(srcs), sssp)
        more = np.concatenate([srcs, srcs + 1, srcs[:1]])[:6] % g.n  # a larger call on the same state
        assert np.array_equal(dg.bfs_batch(more)[:3], bfs) and np.array_equal(dg.sssp_batch(more)[:3], sssp)


@pytest.mark.parametrize("k", [3, 256])
@pytest.mark.parametrize("which", ["teams-bfs", "teams-sssp", "levels", "pull"])
def test_batched_routes_given_up_hold_no_memory(mg, oracle, device, monkeypatch, which, k):
    # after a search that its route could not hold, the graph holds what the general route needs, and of
    # the teams at most 64 MB
    import ctypes as C

    if which.startswith("teams"):
        g = random_graph(mg, 120000, 350000, 3, wmax=20)
    else:
        g = _clique_chain(mg, 60, 20)
        g.values = mg.hash_weights(g, 2, 30)
    srcs = np.resize(np.array([0, g.n // 2, g.n - 1], np.int32), k)
    sssp = which in ("teams-sssp", "pull")
    one = (lambda s: oracle.sssp(g.row_offsets, g.col_idx, g.values, s)) if sssp else (
        lambda s: oracle.bfs(g.row_offsets, g.col_idx, s))
    exp = np.resize(np.stack([one(int(s)) for s in srcs[:3]]), (k, g.n))

    def grown(general):
        with mg.Graph(g, symmetric=True) as dg:
            before = dg.device_bytes()
            if not general:
                for _ in range(2):
                    assert np.array_equal(dg.sssp_batch(srcs) if sssp else dg.bfs_batch(srcs), exp)
            elif which == "levels":  # (a device result needs no rows)
                hip, p, o = C.CDLL("libamdhip64.so"), C.c_void_p(), mg.options(out_on_device=1)
                assert hip.hipMalloc(C.byref(p), C.c_size_t(4 * k * g.n)) == 0
                mg.check(mg.lib().mg_bfs_batch(dg.handle, srcs.ctypes.data_as(C.POINTER(C.c_int32)), k, p, C.byref(o), None))
                hip.hipFree(p)
            else:
                monkeypatch.setenv("MG_FAIL_ALLOC_AT", "1")  # the faster route's first allocation is refused
                assert np.array_equal(dg.sssp_batch(srcs) if sssp else dg.bfs_batch(srcs), exp)
                monkeypatch.delenv("MG_FAIL_ALLOC_AT")
            return dg.device_bytes() - before

    kept = grown(False) - grown(True)
    assert kept == 0 or (which.startswith("teams") and k == 3 and 0 < kept <= 64 << 20)


def _widening(mg, first, doublings):
    """A tree: `first` vertices below the root, then twice as many a level; the last level holds most."""
    src, dst, at, level = [np.zeros(first, np.int64)], [np.arange(1, first + 1)], first + 1, np.arange(1, first + 1)
    for _ in range(doublings):
        kids = np.arange(at, at + 2 * len(level))
        src.append(np.repeat(level, 2)), dst.append(kids)
        at, level = at + len(kids), kids
    g = mg.csr_from_edges(at, np.concatenate(src).astype(np.int32), np.concatenate(dst).astype(np.int32),
                          mg.MG_CSR_SYMMETRIZE | mg.MG_CSR_SORT_COLS)
    g.values = mg.hash_weights(g, 3, 9)
    return g


@pytest.mark.parametrize("sssp", [False, True])
def test_batch_teams_short_of_workgroups_are_tried_again(mg, oracle, device, monkeypatch, sssp):
    # the last level needs most of a team's sixteen workgroups; here teams close with one
    g = _widening(mg, 6, 12)
    srcs = np.zeros(8, np.int32)
    one = oracle.sssp(g.row_offsets, g.col_idx, g.values, 0) if sssp else oracle.bfs(g.row_offsets, g.col_idx, 0)
    o = mg.options(sssp_delta=-1)
    with mg.Graph(g, symmetric=True) as dg:
        monkeypatch.setenv("MG_TEAM_LAUNCH", "1")
        for _ in range(3):
            for row in dg.sssp_batch(srcs, o) if sssp else dg.bfs_batch(srcs):
                assert np.array_equal(row, one)
        monkeypatch.delenv("MG_TEAM_LAUNCH")
        before = dg.device_bytes()
        for row in dg.sssp_batch(np.tile(srcs, 3), o) if sssp else dg.bfs_batch(np.tile(srcs, 3)):
            assert np.array_equal(row, one)
        assert dg.device_bytes() > before  # state for more teams: they took the call


@pytest.mark.parametrize("sssp", [False, True])
def test_batch_teams_beside_a_hub_in_another_component(mg, oracle, device, sssp):
    # a vertex that no team queues in one component; searches of the other one are taken by teams again
    a, b = mg.grid_graph(40, 30, seed=3), mg.grid_graph(50, 40, seed=4)
    n, hub = a.n + b.n + 1500, 7
    src = np.concatenate([np.repeat(np.arange(a.n), np.diff(a.row_offsets)),
                          np.repeat(np.arange(b.n), np.diff(b.row_offsets)) + a.n, np.full(1500, hub)])
    dst = np.concatenate([a.col_idx, b.col_idx + a.n, np.arange(a.n + b.n, n)])
    g = mg.csr_from_edges(n, src.astype(np.int32), dst.astype(np.int32),
                          mg.MG_CSR_SYMMETRIZE | mg.MG_CSR_DEDUPE | mg.MG_CSR_SORT_COLS)
    g.values = mg.hash_weights(g, 3, 9)
    one = (lambda s: oracle.sssp(g.row_offsets, g.col_idx, g.values, s)) if sssp else (
        lambda s: oracle.bfs(g.row_offsets, g.col_idx, s))
    near, far = np.array([0, hub, a.n - 1], np.int32), np.arange(a.n, a.n + 20, dtype=np.int32)
    with mg.Graph(g, symmetric=True) as dg:
        batch = dg.sssp_batch if sssp else dg.bfs_batch
        assert np.array_equal(batch(near), np.stack([one(int(s)) for s in near]))
        before, exp = dg.device_bytes(), np.stack([one(int(s)) for s in far])
        for calls in range(60):
            assert np.array_equal(batch(far), exp)
            if dg.device_bytes() > before:  # state for more teams: they took the call
                break
        assert calls < 59
        assert np.array_equal(batch(near), np.stack([one(int(s)) for s in near]))


@pytest.mark.parametrize("leaves,length", [(1100, 3), (1100, 12), (3000, 9)])
def test_searches_that_alternate_between_teams_and_the_single_workgroup(mg, oracle, device, leaves, length):
    # every star sends a team back; later searches of the graph start from what the earlier ones found
    g = _chain(mg, [length] * 40, [leaves] * 39 + [0], 6)
    with mg.Graph(g, symmetric=True) as dg:
        for src in (0, g.n - 1, g.n // 2, 0, 0):
            assert np.array_equal(dg.bfs(src), oracle.bfs(g.row_offsets, g.col_idx, src))
            assert np.array_equal(dg.sssp(src), oracle.sssp(g.row_offsets, g.col_idx, g.values, src))


def test_a_search_needs_no_memory_for_its_team(mg, oracle, device, monkeypatch):
    g = mg.grid_graph(90, 70, seed=2, weight_max=16)
    with mg.Graph(g, symmetric=True) as dg:
        dg.sssp(0, mg.options(iter_num=2))  # (the tasks of the dense levels, made by the first search)
        for fn, exp in ((dg.bfs, oracle.bfs(g.row_offsets, g.col_idx, 0)),
                        (dg.sssp, oracle.sssp(g.row_offsets, g.col_idx, g.values, 0))):
            monkeypatch.setenv("MG_FAIL_ALLOC_AT", "1")
            assert np.array_equal(fn(0), exp)
            monkeypatch.delenv("MG_FAIL_ALLOC_AT")


def test_batch_pull_sizes_that_share_a_row_width(mg, oracle, device):
    # larger and smaller calls in turn on one graph, as many columns as the width has and one
    g = random_graph(mg, 1501, 12000, 6, wmax=30)
    srcs = np.random.default_rng(1).integers(0, g.n, 64).astype(np.int32)
    exp = np.stack([oracle.sssp(g.row_offsets, g.col_idx, g.values, int(s)) for s in srcs])
    with mg.Graph(g, symmetric=True) as dg:
        for k in (1, 32, 3, 31, 32, 4, 33, 64, 35, 64, 5):
            for lo in (0, 64 - k):
                assert np.array_equal(dg.sssp_batch(srcs[lo:lo + k]), exp[lo:lo + k]), (k, lo)


def test_the_tuner_keeps_no_bucket_width_for_a_pulled_batch(mg, device):
    g = mg.rmat_graph(12, 16, seed=3, weight_max=64)
    with mg.Graph(g, symmetric=True) as dg:
        for start in (0, 7):
            for _ in range(3):
                best, _ = dg.autotune("sssp_batch", mg.pick_sources(g, 4, seed=1), start=mg.options(sssp_delta=start), reps=1)
                assert best.sssp_delta == start


@pytest.mark.parametrize("symmetric", [False, True])
@pytest.mark.parametrize("n", [255, 257, 65537, 262145, 524321])
def test_frontier_slices_of_the_general_batches(mg, oracle, device, monkeypatch, n, symmetric):
    # as above for both directions, with batches on the shared frontier: the memory of the other route
    # for sparse graphs is refused
    g = random_graph(mg, n, 3 * n if symmetric else 6 * n, seed=n + 1, symmetric=symmetric, wmax=16)
    assert g.m < 8 * n
    srcs = np.array([int(np.argmax(g.degrees())), n - 1, 0], np.int32)
    bfs = [oracle.bfs(g.row_offsets, g.col_idx, int(s)) for s in srcs]
    sssp = [oracle.sssp(g.row_offsets, g.col_idx, g.values, int(s)) for s in srcs]
    with mg.Graph(g, symmetric=symmetric) as dg:
        assert np.array_equal(dg.bfs(int(srcs[0])), bfs[0]) and np.array_equal(dg.sssp(int(srcs[0])), sssp[0])
        for batch, exp, at in ((dg.bfs_batch, bfs, "1"), (dg.sssp_batch, sssp, "01")):
            before = dg.device_bytes()
            monkeypatch.setenv("MG_FAIL_ALLOC_AT", at)  # the first allocation from here on
            for got, row in zip(batch(srcs), exp):
                assert np.array_equal(got, row)
            monkeypatch.delenv("MG_FAIL_ALLOC_AT")
            assert dg.device_bytes() >= before + 4 * mg.MG_BATCH_MAX * n  # the general route's rows


def test_device_bytes_beside_calls_that_release_state(mg, oracle, device):
    # asked for from another thread while batches make, grow and release their routes' state
    import threading

    g = _clique_chain(mg, 60, 20)
    g.values = mg.hash_weights(g, 2, 30)
    sparse = random_graph(mg, 120000, 350000, 3, wmax=20)
    stop, seen = threading.Event(), []
    with mg.Graph(g, symmetric=True) as a, mg.Graph(sparse, symmetric=True) as b:
        def ask():
            while not stop.is_set():
                seen.extend((a.device_bytes(), b.device_bytes()))

        t = threading.Thread(target=ask)
        t.start()
        for k in (1, 40, 100):
            srcs = np.arange(k, dtype=np.int32)
            for dg, h in ((a, g), (b, sparse)):
                assert np.array_equal(dg.sssp_batch(srcs)[0], oracle.sssp(h.row_offsets, h.col_idx, h.values, 0))
                assert np.array_equal(dg.bfs_batch(srcs)[-1], oracle.bfs(h.row_offsets, h.col_idx, k - 1))
        stop.set()
        t.join()
    assert seen and min(seen) > 0 and max(seen) < 1 << 34
