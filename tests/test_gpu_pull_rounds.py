"""Traversals whose rounds pull (a run from scratch on 2^18 edges or more): SSSP and BFS
equal the unique fixed point bit for bit, distances and smallest-id parents; SSWP widths
equal it and its parents are valid and acyclic.  Graphs: R-MAT, rows across many 1024-edge
tiles, tiles that run over tens of thousands of empty rows (the per-edge search), a
frontier that grows and shrinks around the switch between push and pull, and one that
stays small for longer than the first group of rounds."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu
INF = 0xFFFFFFFF


def csr(n, u, v, rng, wmax):
    key = np.unique(u.astype(np.int64) * n + v.astype(np.int64))
    u, v = key // n, key % n
    u, v = u[u != v], v[u != v]
    off = np.zeros(n + 1, np.uint64)
    off[1:] = np.cumsum(np.bincount(u, minlength=n))
    return off, v.astype(np.uint32), rng.integers(1, wmax + 1, len(u)).astype(np.uint32), u, v


def graph(name, rng):
    if name == "rmat":
        g = oracle.Graph.rmat(16, 16, seed=3, weights="u32", wmin=1, wmax=64)
        off, col, w = g.csr()
        u = np.repeat(np.arange(g.n), np.diff(off.astype(np.int64)))
        return g.n, off, col, w, u, col.astype(np.int64)
    if name == "hubs":  # 40 destinations with up to 30,000 in-edges each, and the way back out
        n = 60_000
        u = np.concatenate([rng.integers(0, n, 300_000), rng.integers(0, 40, 120_000), np.zeros(200, int)])
        v = np.concatenate([(40 * rng.random(300_000) ** 2).astype(int), rng.integers(0, n, 120_000),
                            rng.integers(0, n, 200)])
    elif name == "gaps":  # in-edges at both ends of the ids only, one tile over the 94,000 between
        n = 100_001
        ends = np.concatenate([np.arange(0, 3000), np.arange(n - 3000, n)])
        u, v = rng.choice(ends, 330_000), rng.choice(ends, 330_000)
        u[:300], v[:300] = 0, rng.choice(ends, 300)
    elif name == "late":  # a path of 150 into a core: rounds enqueued without pulls meet the core's frontier
        n = 30_150
        core = 150 + rng.integers(0, n - 150, (2, 300_000))
        u, v = np.concatenate([np.arange(150), core[0]]), np.concatenate([np.arange(1, 151), core[1]])
    else:  # layers: 5 vertices, then 200, 20,000, 20,000, 50, 20,000, 10
        sizes = [1, 5, 200, 20_000, 20_000, 50, 20_000, 10]
        n = sum(sizes)
        at = np.concatenate([[0], np.cumsum(sizes)])
        us, vs = [], []
        for k in range(len(sizes) - 1):
            e = 12 * max(sizes[k], sizes[k + 1])
            us.append(at[k] + rng.integers(0, sizes[k], e))
            vs.append(at[k + 1] + rng.integers(0, sizes[k + 1], e))
        u, v = np.concatenate(us), np.concatenate(vs)
    off, col, w, u, v = csr(n, u, v, rng, 64)
    return n, off, col, w, u, v


def relax(n, u, v, w, app):
    """Words of the fixed point by full relaxation: distances, hops or ~widths."""
    d = np.full(n, INF, np.int64)
    d[0] = 0
    while True:
        if app == "sswp":
            c = INF - np.minimum(INF - d[u], w.astype(np.int64))
        else:
            c = d[u] + (1 if app == "bfs" else w.astype(np.int64))
        c[d[u] >= INF] = INF
        new = d.copy()
        np.minimum.at(new, v, np.minimum(c, INF))
        if np.array_equal(new, d):
            return d, c
        d = new


@pytest.mark.parametrize("app", ["sssp", "bfs", "sswp"])
@pytest.mark.parametrize("name", ["rmat", "hubs", "gaps", "late", "layers"])
def test_pull_rounds_reach_the_fixed_point(gpu, name, app):
    n, off, col, w, u, v = graph(name, np.random.default_rng(4))
    assert len(col) >= 1 << 18
    d, c = relax(n, u, v, w, app)
    code = {"sssp": gpu.APP_SSSP, "bfs": gpu.APP_BFS, "sswp": gpu.APP_SSWP}[app]
    with gpu.Context() as ctx:
        ctx.upload_csr(off, col, w)
        ctx.traversal_init(code, 0)
        st = ctx.sssp_run()
        val, par = ctx.sssp_download()
        ctx.traversal_init(code, 0)  # the lists and bitmaps are as a first run leaves them
        ctx.sssp_run()
        val2, par2 = ctx.sssp_download()
        ctx.traversal_init(code, 0)  # and a loop of single (push) rounds agrees
        while ctx.sssp_step():
            pass
        val3, par3 = ctx.sssp_download()
    assert st["pull_rounds"] >= 1 and st["pull_rounds"] + st["push_rounds"] == st["rounds"]
    word = INF - val.astype(np.int64) if app == "sswp" else val.astype(np.int64)
    assert np.array_equal(word, d)
    assert np.array_equal(val, val2) and np.array_equal(val, val3)
    reached = (d < INF) & (np.arange(n) > 0)
    if app != "sswp":
        best = np.full(n, n, np.int64)
        tie = (c == d[v]) & (c < INF)
        np.minimum.at(best, v[tie], u[tie])
        assert np.array_equal(par[reached], best[reached])
        assert np.array_equal(par, par2) and np.array_equal(par, par3)
        return
    # an edge from the parent gives the width, and the parents lead to the source
    ok = np.zeros(n, bool)
    tie = (c == d[v]) & (par[v] == u)
    ok[v[tie]] = True
    assert ok[reached].all()
    up = np.where(reached, par, 0).astype(np.int64)
    for _ in range(int(n).bit_length()):
        up = up[up]
    assert (up[reached] == 0).all()


@pytest.mark.parametrize("app", ["sssp", "bfs"])
def test_a_run_without_pulls_before_one_with_them(gpu, app):
    """After a run from scratch that had no pull, the next one's rounds are enqueued
    without, until its frontier asks for one; at a round cap on either side of that too."""
    n, off, col, w, u, v = graph("late", np.random.default_rng(6))
    code = {"sssp": gpu.APP_SSSP, "bfs": gpu.APP_BFS}[app]
    with gpu.Context() as ctx:
        ctx.upload_csr(off, col, w)

        def run(source, cap=0):
            ctx.set_params(max_rounds=cap or 100000)
            ctx.traversal_init(code, source)
            try:
                st = ctx.sssp_run()
            except gpu.SumincError as e:
                assert e.code == gpu.E_NOT_CONVERGED
                st = ctx.stats()
            return st, *ctx.sssp_download()

        first = run(150)
        assert first[0]["pull_rounds"] > 0
        ctx.set_params(max_rounds=20)
        caps = {}
        for cap in (1, 2, 3, 4, 5, 7):
            caps[cap] = run(150, cap)
        for cap in caps:
            assert run(0, 40)[0]["pull_rounds"] == 0  # on the path only: no pull
            st, val, par = run(150, cap)
            assert st["rounds"] == min(cap, first[0]["rounds"])
            # (a capped SSSP's words depend on the order of the round; BFS' do not)
            if app == "bfs":
                assert np.array_equal(val, caps[cap][1])
            assert run(0, 40)[0]["pull_rounds"] == 0
            st, val, par = run(150)
            assert st["pull_rounds"] > 0 and st["pull_rounds"] + st["push_rounds"] == st["rounds"]
            assert np.array_equal(val, first[1]) and np.array_equal(par, first[2])


def test_widths_with_many_ties_keep_a_tree_of_parents(gpu):
    """SSWP on three widths: rows of 10,000 in-edges, each over many tiles and nearly all
    of them ties, from scratch and after a batch that deletes every hub's parent edge."""
    rng = np.random.default_rng(8)
    n, hubs = 50_000, 60
    u = np.concatenate([rng.integers(0, n, 600_000), rng.integers(0, hubs, 200_000), np.zeros(60, int)])
    v = np.concatenate([rng.integers(0, hubs, 600_000), rng.integers(0, n, 200_000), rng.integers(0, n, 60)])
    off, col, w, u, v = csr(n, u, v, rng, 3)

    def check(val, par, u, v, w):
        d, c = relax(n, u, v, w, "sswp")
        assert np.array_equal(INF - val.astype(np.int64), d)
        reached = (d < INF) & (np.arange(n) > 0)
        ok = np.zeros(n, bool)
        ok[v[(c == d[v]) & (par[v] == u)]] = True
        assert ok[reached].all()
        up = np.where(reached, par, 0).astype(np.int64)
        for _ in range(int(n).bit_length()):
            up = up[up]
        assert (up[reached] == 0).all()

    with gpu.Context() as ctx:
        ctx.upload_csr(off, col, w)
        ctx.traversal_init(gpu.APP_SSWP, 0)
        assert ctx.sssp_run()["pull_rounds"] >= 1
        val, par = ctx.sssp_download()
        check(val, par, u, v, w)
        gone = np.isin(u * n + v, [int(par[h]) * n + h for h in range(1, hubs)])
        rec = np.zeros(gone.sum(), gpu.UPDATE_DTYPE)
        rec["type"], rec["u"], rec["v"] = 1, u[gone], v[gone]
        assert len(rec) > hubs // 2
        ctx.apply_batch(rec)
        ctx.sssp_run()
        val, par = ctx.sssp_download()
        check(val, par, u[~gone], v[~gone], w[~gone])
