"""Extrapolated delta series: wherever a run stops, rank and delta are a state of the
same fixed point, r + (I - M)^-1 delta, and these graphs take no more rounds than plain
ones (one more where sums may cross T a round later).

Graphs: ones whose series lines up with one eigenvector (R-MAT, uniform, communities),
ones that are eigenvectors from the start (ring, pairs) and ones that never line up
(signed mass on a grid, a path, a ring), below and above a block of 1024 vertices.

Tolerances against scipy's sparse solve: the stop rule's residual / (1 - d), plus rounding.
FP64: 1e-12 of the state's mass.  FP32: a round rounds every delta to 2^-24, an
extrapolation amplifies that by 1 + 2 beta <= 99 once, and (I - M)^-1 by 1 / (1 - d):
2^-24 * (rounds + 99) / 0.15 of the mass at most, 1e-5 of it over 40 rounds and less
where deltas shrink.
"""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as sla

from tests.conftest import DAMPING

pytestmark = pytest.mark.gpu


def graph(name):
    rng = np.random.default_rng(7)
    if name == "one":
        n, u, v = 1, [], []
    elif name == "ring":
        n = 1025
        u = np.arange(n)
        v = (u + 1) % n
    elif name == "pairs":
        n = 1024
        u = np.arange(n)
        v = u ^ 1
    elif name == "path":
        n = 700
        u = np.arange(n - 1)
        v = u + 1
    elif name == "grid":
        a = 37
        n = a * a
        x, y = [t.ravel() for t in np.meshgrid(np.arange(a), np.arange(a))]
        u = np.concatenate([(x * a + y)[(0 <= x + dx) & (x + dx < a) & (0 <= y + dy) & (y + dy < a)]
                            for dx, dy in ((1, 0), (-1, 0), (0, 1), (0, -1))])
        v = np.concatenate([((x + dx) * a + y + dy)[(0 <= x + dx) & (x + dx < a) & (0 <= y + dy) & (y + dy < a)]
                            for dx, dy in ((1, 0), (-1, 0), (0, 1), (0, -1))])
    elif name == "communities":
        n, c = 5000, 100
        u = rng.integers(0, n, 8 * n)
        v = np.where(rng.random(8 * n) < 0.98, u // c * c + rng.integers(0, c, 8 * n), rng.integers(0, n, 8 * n))
    elif name == "uniform":
        n = 3001
        u, v = rng.integers(0, n, 6 * n), rng.integers(0, n, 6 * n)
    else:  # skewed ids, many vertices without out-edges
        n = 4099
        u, v = (n * rng.random(8 * n) ** 4).astype(int), (n * rng.random(8 * n) ** 3).astype(int)
    key = np.unique(np.asarray(u, np.int64) * n + np.asarray(v, np.int64))
    u, v = key // n, key % n
    u, v = u[u != v], v[u != v]
    off = np.zeros(n + 1, np.uint64)
    off[1:] = np.cumsum(np.bincount(u, minlength=n))
    return n, u, v, off


def system(n, u, v):
    deg = np.bincount(u, minlength=n) if len(u) else np.zeros(n)
    return sp.csr_matrix((DAMPING / deg[u], (v, u)), shape=(n, n)) if len(u) else sp.csr_matrix((n, n))


def plain_rounds(M, x, T):
    """Rounds of the series with the activity rule: |delta| <= T / n waits."""
    k = 0
    while np.abs(x).sum() >= T:
        a = np.where(np.abs(x) > T / len(x), x, 0.0)
        x, k = x - a + M @ a, k + 1
    return k


def limit(M, r, x):
    return r + sla.spsolve(sp.eye(M.shape[0], format="csc") - M.tocsc(), x)


def series_limit(M, x):
    """The same for larger graphs, whose factors fill in: the series to 2^-60."""
    r = x.copy()
    while np.abs(x).sum() > 1e-18:
        x = M @ x
        r += x
    return r


GRAPHS = ["one", "ring", "pairs", "path", "grid", "communities", "uniform", "skewed"]


@pytest.mark.parametrize("seed", ["uniform", "vertex", "signed"])
@pytest.mark.parametrize("name", GRAPHS)
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_run_reaches_the_fixed_point(gpu, prec, name, seed):
    n, u, v, off = graph(name)
    M = system(n, u, v)
    x = np.full(n, (1 - DAMPING) / n)
    if seed == "vertex":
        x = np.zeros(n)
        x[0] = 1 - DAMPING
    elif seed == "signed":
        x = np.random.default_rng(3).standard_normal(n)
        x *= 0.1 / np.abs(x).sum()
    T = 1e-11 if prec == "fp64" else 1e-7
    p = gpu.PR_FP64 if prec == "fp64" else gpu.PR_FP32_KAHAN
    want = limit(M, np.zeros(n), x)
    with gpu.Context(pr_precision=p, termcheck_threshold=T, max_rounds=1000) as ctx:
        ctx.upload_csr(off, v.astype(np.uint32))
        ctx.pr_upload(np.zeros(n), x)
        st = ctx.pr_run()
        r, d = ctx.pr_download()
    mass = np.abs(x).sum()
    assert st["residual"] < T
    assert np.isclose(np.abs(d).sum(), st["residual"], rtol=1e-5, atol=T * 1e-5)
    # one round more: FP32 sums may cross T a round later
    assert st["rounds"] <= plain_rounds(M, x, T) + 1
    assert np.abs(r - want).sum() <= T / (1 - DAMPING) + mass * (1e-12 if prec == "fp64" else 1e-5)


@pytest.mark.parametrize("name", ["ring", "communities", "uniform", "skewed"])
@pytest.mark.parametrize("cap", [1, 2, 3, 5, 6, 8, 9, 10, 11, 12, 14])
def test_round_cap_leaves_a_state_of_the_same_fixed_point(gpu, name, cap):
    n, u, v, off = graph(name)
    M = system(n, u, v)
    x = np.full(n, (1 - DAMPING) / n)
    want = limit(M, np.zeros(n), x)
    with gpu.Context(pr_precision=gpu.PR_FP64, termcheck_threshold=1e-11, max_rounds=cap) as ctx:
        ctx.upload_csr(off, v.astype(np.uint32))
        ctx.pr_init()
        st = ctx.pr_run(allow_not_converged=True)
        r, d = ctx.pr_download()
        # the (untaken) rest of an inactive vertex stays in delta, so the state is exact
        assert np.abs(limit(M, r, d) - want).sum() < 1e-12
        assert np.abs(d).sum() <= (1 - DAMPING) * DAMPING ** st["rounds"] * (1 + 1e-9)
        if (name, cap) in (("communities", 6), ("ring", 2), ("ring", 3)):
            # the decision at the cap itself chose a step: far below as many plain rounds
            assert np.abs(d).sum() < 0.1 * (1 - DAMPING) * DAMPING ** cap
        ctx.set_params(max_rounds=1000)
        ctx.pr_run()
        r, _ = ctx.pr_download()
    assert np.abs(r - want).sum() <= 1e-11 / (1 - DAMPING) + 1e-12


@pytest.mark.parametrize("name,n", [("uniform", 3001), ("skewed", 4099), ("uniform", 1500)])
@pytest.mark.parametrize("T", [1e-2, 1e-4, 1e-6, 1e-9, 1e-11])
def test_runs_that_line_up_take_steps(gpu, name, n, T):
    """On graphs whose series lines up the rounds fall well below plain ones', the last
    decision takes a step too (the residual is below what the rounds alone reach), and the
    state it leaves is exact.  1500 vertices: in one workgroup."""
    n, u, v, off = graph(name) if n > 2048 else uniform(n)
    M = system(n, u, v)
    x = np.full(n, (1 - DAMPING) / n)
    want = limit(M, np.zeros(n), x)
    with gpu.Context(pr_precision=gpu.PR_FP64, termcheck_threshold=T, max_rounds=1000) as ctx:
        ctx.upload_csr(off, v.astype(np.uint32))
        ctx.pr_init()
        st = ctx.pr_run()
        r, d = ctx.pr_download()
    plain = plain_rounds(M, x, T)
    assert st["rounds"] <= 0.4 * plain + 1
    k, y = 0, x
    while k < st["rounds"]:
        y, k = M @ y, k + 1
    assert st["residual"] < T < 0.5 * np.abs(y).sum()
    assert np.abs(limit(M, r, d) - want).sum() < 1e-12


def uniform(n):
    rng = np.random.default_rng(n)
    key = np.unique(rng.integers(0, n, 6 * n) * n + rng.integers(0, n, 6 * n))
    u, v = key // n, key % n
    u, v = u[u != v], v[u != v]
    off = np.zeros(n + 1, np.uint64)
    off[1:] = np.cumsum(np.bincount(u, minlength=n))
    return n, u, v, off


def hubs(n=6007, hubs=300):
    """A skewed core over `hubs` vertices; the others hang on one of them, most both ways."""
    rng = np.random.default_rng(11)
    u, v = (hubs * rng.random(8 * hubs) ** 2).astype(int), (hubs * rng.random(8 * hubs) ** 2).astype(int)
    leaf = np.arange(hubs, n)
    h = rng.integers(0, hubs, len(leaf))
    back = rng.random(len(leaf)) < 0.8
    key = np.unique(np.concatenate([u * n + v, leaf * n + h, (h * n + leaf)[back]]).astype(np.int64))
    u, v = key // n, key % n
    u, v = u[u != v], v[u != v]
    off = np.zeros(n + 1, np.uint64)
    off[1:] = np.cumsum(np.bincount(u, minlength=n))
    return n, u, v, off


@pytest.mark.parametrize("div", [3, 1_000_000, 0], ids=["mixed", "pull", "push"])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_sketch_run_reaches_the_fixed_point(gpu, prec, div):
    """From scratch, from a signed state and at round caps, over supernodes: the exits'
    and entries' share of an extrapolation step (pull rounds), and none of it (push)."""
    n, u, v, off = hubs()
    M = system(n, u, v)
    T = 1e-11 if prec == "fp64" else 1e-7
    tol = 1e-12 if prec == "fp64" else 1e-5
    p = gpu.PR_FP64 if prec == "fp64" else gpu.PR_FP32_KAHAN
    x0 = np.full(n, (1 - DAMPING) / n)
    x1 = np.random.default_rng(5).standard_normal(n)
    x1 *= 0.1 / np.abs(x1).sum()
    with gpu.Context(pr_precision=p, termcheck_threshold=T, max_rounds=1000, pull_threshold_div=div) as ctx:
        ctx.upload_csr(off, v.astype(np.uint32))
        ctx.cluster_leaves(1024, 2)
        for x in (x0, x1):
            info = ctx.sum_build(2, 1024, 1.0)  # a fresh build: every cluster runs its precompute
            assert info["clusters"] > 100 and info["entries"] > 100
            want = limit(M, np.zeros(n), x)
            ctx.pr_upload(np.zeros(n), x)
            st = ctx.sum_pr_run()
            r, _ = ctx.pr_download()
            assert st["residual"] < T
            assert st["sketch_rounds"] + st["residual_rounds"] <= plain_rounds(M, x, T) + 3
            assert np.abs(r - want).sum() <= T / (1 - DAMPING) + 0.15 * tol
        want = limit(M, np.zeros(n), x0)
        for cap in (4, 7, 9, 12):
            ctx.set_params(max_rounds=cap)
            ctx.pr_upload(np.zeros(n), x0)
            try:
                ctx.sum_pr_run()
            except gpu.SumincError as e:
                assert e.code == gpu.E_NOT_CONVERGED
            r, d = ctx.pr_download()
            assert np.abs(limit(M, r, d) - want).sum() <= 0.15 * tol


def test_sketch_rounds_take_steps_when_they_pull(gpu):
    """Pulling sketch rounds that line up extrapolate (fewer rounds than pushing ones, which
    do not), up to the decision that ends the phase, and every threshold leaves an exact
    state: the entries', the exits' and the Singles' share of the last step."""
    n, u, v, off = hubs()
    M = system(n, u, v)
    x = np.full(n, (1 - DAMPING) / n)
    want = limit(M, np.zeros(n), x)
    rounds = {}
    for div in (1_000_000, 0):
        with gpu.Context(pr_precision=gpu.PR_FP64, max_rounds=1000, pull_threshold_div=div) as ctx:
            ctx.upload_csr(off, v.astype(np.uint32))
            ctx.cluster_leaves(1024, 2)
            for T in (1e-2, 1e-3, 1e-4, 1e-5, 1e-6, 1e-7, 1e-8):
                ctx.set_params(termcheck_threshold=T)
                ctx.sum_build(2, 1024, 1.0)
                ctx.pr_upload(np.zeros(n), x)
                rounds[div, T] = ctx.sum_pr_run()["sketch_rounds"]
                r, d = ctx.pr_download()
                assert np.abs(limit(M, r, d) - want).sum() < 1e-12
                assert np.abs(d).sum() < T
    for T in (1e-2, 1e-3, 1e-4, 1e-5, 1e-6, 1e-7, 1e-8):
        assert rounds[1_000_000, T] <= 0.65 * rounds[0, T]


@pytest.mark.parametrize("T", [1e-3, 1e-6, 1e-9])
@pytest.mark.parametrize("big", [False, True], ids=["one_turn", "decide"])
def test_weighted_series_that_line_up_take_steps(gpu, T, big):
    """Rounds well below plain ones', and what the series leaves out is its residual's
    share, which holds only if the step that ended it is in the result (2^18 + 1 vertices:
    decided by a launch of its own)."""
    n, u, v, off = uniform((1 << 18) + 1 if big else 3001)
    w = (1.0 - np.random.default_rng(1).random(len(u))).astype(np.float32)
    s = np.bincount(u, weights=w.astype(float), minlength=n)
    M = sp.csr_matrix((DAMPING * w.astype(float) / s[u], (v, u)), shape=(n, n))
    p = np.full(n, 1.0 / n, np.float32)
    c = np.random.default_rng(2).random(n).astype(np.float32) + 0.5
    x = (1 - DAMPING) * p.astype(float)
    with gpu.Context(pr_precision=gpu.PR_FP64, termcheck_threshold=T, max_rounds=1000) as ctx:
        ctx.upload_csr(off, v.astype(np.uint32), w)
        ctx.wpr_set_weights(w)
        _, st = ctx.wpr_forward(p)
        r, _ = ctx.wpr_download()
        _, _, sb = ctx.wpr_backward(c)
        _, lam = ctx.wpr_download(adjoint=True)
    assert st["rounds"] <= 0.5 * plain_rounds_all(M, x, T) + 1
    assert sb["rounds"] <= 0.5 * plain_rounds_all(M.T.tocsr(), c.astype(float), T * np.abs(c).sum()) + 1
    left = DAMPING / (1 - DAMPING)
    assert np.abs(r - series_limit(M, x)).sum() <= left * st["residual"] * (1 + 1e-6) + 1e-12
    # (d W contracts the maximum norm; on this graph the 1-norm grows by 2 at most)
    assert np.abs(lam - series_limit(M.T.tocsr(), c.astype(float))).sum() <= 2 * left * sb["residual"] + 1e-9


@pytest.mark.parametrize("name", ["ring", "path", "grid", "communities", "uniform", "skewed"])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_weighted_series_and_adjoint(gpu, prec, name):
    """Forward from one vertex and adjoint from signed loss weights (the transpose does
    not contract the 1-norm) against solves of both systems."""
    n, u, v, off = graph(name)
    rng = np.random.default_rng(9)
    w = (1.0 - rng.random(len(u))).astype(np.float32)
    s = np.bincount(u, weights=w.astype(float), minlength=n)
    M = sp.csr_matrix((DAMPING * w.astype(float) / s[u], (v, u)), shape=(n, n))
    p = np.zeros(n, np.float32)
    p[0] = 1.0
    c = rng.standard_normal(n).astype(np.float32)
    T = 1e-11 if prec == "fp64" else 1e-7
    tol = 1e-6 if prec == "fp64" else 1e-5  # rank and gradients come back as FP32
    pr = gpu.PR_FP64 if prec == "fp64" else gpu.PR_FP32_KAHAN
    with gpu.Context(pr_precision=pr, termcheck_threshold=T, max_rounds=2000) as ctx:
        ctx.upload_csr(off, v.astype(np.uint32), w)
        ctx.wpr_set_weights(w)
        r, st = ctx.wpr_forward(p)
        gp, gw, sb = ctx.wpr_backward(c)
    want = limit(M, np.zeros(n), (1 - DAMPING) * p.astype(float))
    lam = limit(M.T.tocsr(), np.zeros(n), c.astype(float))
    assert st["rounds"] <= max(1, plain_rounds_all(M, (1 - DAMPING) * p.astype(float), T)) + 1
    assert sb["rounds"] <= max(1, plain_rounds_all(M.T.tocsr(), c.astype(float), T * np.abs(c).sum())) + 1
    assert np.abs(r - want).sum() <= T / (1 - DAMPING) + tol
    gw_want = (want / np.where(s > 0, s, 1))[u] * (DAMPING * lam[v] - (M.T @ lam)[u])
    assert np.abs(gp - (1 - DAMPING) * lam).max() <= tol * np.abs(lam).max()
    assert np.abs(gw - gw_want).max() <= tol * max(np.abs(gw_want).max(), np.abs(lam).max() * (want[u] / s[u]).max())


@pytest.mark.parametrize("n", [1024, 1025, 1 << 18, (1 << 18) + 1])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_weighted_series_around_one_partial_a_thread(gpu, prec, n):
    """Up to 2^18 vertices the step's workgroups decide for themselves, beyond a launch of
    its own does: the same series, also where the round cap ends it."""
    rng = np.random.default_rng(n)
    u, v = rng.integers(0, n, 3 * n), rng.integers(0, n, 3 * n)
    key = np.unique(u * n + v)
    u, v = key // n, key % n
    u, v = u[u != v], v[u != v]
    off = np.zeros(n + 1, np.uint64)
    off[1:] = np.cumsum(np.bincount(u, minlength=n))
    w = (1.0 - rng.random(len(u))).astype(np.float32)
    s = np.bincount(u, weights=w.astype(float), minlength=n)
    M = sp.csr_matrix((DAMPING * w.astype(float) / s[u], (v, u)), shape=(n, n))
    p = rng.random(n).astype(np.float32) / n
    c = rng.standard_normal(n).astype(np.float32)
    T = 1e-11 if prec == "fp64" else 1e-7
    pr = gpu.PR_FP64 if prec == "fp64" else gpu.PR_FP32_KAHAN
    x = (1 - DAMPING) * p.astype(float)
    with gpu.Context(pr_precision=pr, termcheck_threshold=T, max_rounds=2000) as ctx:
        ctx.upload_csr(off, v.astype(np.uint32), w)
        ctx.wpr_set_weights(w)
        for _ in range(2):  # the second run's first group is what the first one took
            r, st = ctx.wpr_forward(p)
            gp, _, sb = ctx.wpr_backward(c)
        assert 1 < st["rounds"] <= plain_rounds_all(M, x, T) + 1 and st["residual"] < T
        assert 1 < sb["rounds"] <= plain_rounds_all(M.T.tocsr(), c.astype(float), T * np.abs(c).sum()) + 1
        ctx.set_params(max_rounds=5)
        with pytest.raises(gpu.SumincError) as e:
            ctx.wpr_forward(p)
        assert e.value.code == gpu.E_NOT_CONVERGED
        ctx.set_params(max_rounds=2000)
        again, st2 = ctx.wpr_forward(p)
    assert st2["rounds"] == st["rounds"]
    want = series_limit(M, x)
    tol = 1e-6 if prec == "fp64" else 1e-5  # rank and gradients come back as FP32
    assert np.abs(r - want).sum() <= T / (1 - DAMPING) + tol
    assert np.abs(again - want).sum() <= T / (1 - DAMPING) + tol
    lam = series_limit(M.T.tocsr(), c.astype(float))
    assert np.abs(gp - (1 - DAMPING) * lam).max() <= tol * np.abs(lam).max()


def plain_rounds_all(M, x, T):
    k = 0
    while np.abs(x).sum() >= T:
        x, k = M @ x, k + 1
    return k


@pytest.mark.parametrize("n,m", [(2048, 32768), (2048, 32769), (2049, 32768), (2, 1), (1024, 1), (33, 1000)])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_runs_at_the_edge_of_one_workgroup(gpu, n, m, prec):
    """Graphs of up to 2048 vertices and 32768 edges run in one workgroup, 512 rounds a
    launch: at its limits and just beyond, to the fixed point and over 1100 rounds."""
    rng = np.random.default_rng(n + m)
    key = np.unique((n * rng.random(8 * m) ** 2).astype(np.int64) * n + rng.integers(0, n, 8 * m))
    key = key[key // n != key % n]
    key = np.sort(rng.permutation(key)[:m])
    assert len(key) == min(m, n * (n - 1))
    u, v = key // n, key % n
    off = np.zeros(n + 1, np.uint64)
    off[1:] = np.cumsum(np.bincount(u, minlength=n))
    M = system(n, u, v)
    x = np.full(n, (1 - DAMPING) / n)
    want = limit(M, np.zeros(n), x)
    T = 1e-11 if prec == "fp64" else 1e-7
    p = gpu.PR_FP64 if prec == "fp64" else gpu.PR_FP32_KAHAN
    with gpu.Context(pr_precision=p, termcheck_threshold=T, max_rounds=1000) as ctx:
        ctx.upload_csr(off, v.astype(np.uint32))
        ctx.pr_init()
        st = ctx.pr_run()
        r, d = ctx.pr_download()
        assert st["residual"] < T and st["pull_rounds"] + st["push_rounds"] == st["rounds"]
        assert np.abs(r - want).sum() <= T / (1 - DAMPING) + 0.15 * (1e-12 if prec == "fp64" else 1e-5)
        assert abs(st["mass_defect"]) <= (1e-13 if prec == "fp64" else 1e-6)
        if prec == "fp64" and m > 1000:
            ctx.set_params(termcheck_threshold=0.0, max_rounds=1100)
            ctx.pr_init()
            st = ctx.pr_run(allow_not_converged=True)
            r, d = ctx.pr_download()
            assert st["rounds"] == 1100
            assert np.abs(limit(M, r, d) - want).sum() <= 1e-13


@pytest.mark.parametrize("div", [3, 1_000_000, 0], ids=["mixed", "pull", "push"])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_reseed_keeps_the_fixed_point(gpu, prec, div):
    """After a batch rank and delta are a state of the new graph's fixed point: sources
    that lose all edges, gain their first, swap edges at the same degree, only change
    weights, or are named by deletes of nothing; also after a batch without pulls
    between two with them (the pull's columns are not carried over it)."""
    n, u, v, off = hubs()
    rng = np.random.default_rng(21)
    p = gpu.PR_FP64 if prec == "fp64" else gpu.PR_FP32_KAHAN
    T = 1e-11 if prec == "fp64" else 1e-7
    tol = 0.15 * (1e-12 if prec == "fp64" else 1e-5)
    have = set(zip(u.tolist(), v.tolist()))

    def ops(k):
        deg = np.bincount([a for a, _ in have], minlength=n)
        out = []
        some = sorted(have)
        lose = rng.choice(np.flatnonzero((deg > 0) & (deg < 4)), 40, replace=False)
        for a in lose:  # every edge of some sources goes
            out += [(1, a, b) for x, b in some if x == a]
        none = np.flatnonzero(deg == 0)  # (from the second batch on: the first makes some)
        for a in rng.choice(none, min(30, len(none)), replace=False) if len(none) else []:  # first edges
            out += [(0, a, int(b)) for b in rng.integers(0, 300, 2) if b != a]
        for i in rng.choice(len(some), 60, replace=False):  # an edge for another: the same degree
            a, b = some[i]
            c = int(rng.integers(0, n))
            out += [(1, a, b)] + ([(0, a, c)] if c != a and (a, c) not in have else [])
        for i in rng.choice(len(some), 20, replace=False):  # an add of an edge that is there
            out.append((0, *some[i]))
        for a, b in rng.integers(0, n, (20, 2)):  # a delete of one that is not
            if (a, b) not in have and a != b:
                out.append((1, int(a), int(b)))
        rec = np.zeros(len(out), gpu.UPDATE_DTYPE)
        rec["type"], rec["u"], rec["v"] = np.array(out).T
        adds = {(a, b) for t, a, b in out if t == 0}
        return rec, (have - {(a, b) for t, a, b in out if t == 1}) | adds

    with gpu.Context(pr_precision=p, termcheck_threshold=T, max_rounds=1000, pull_threshold_div=div,
                     pull_compact_kib=1) as ctx:
        ctx.upload_csr(off, v.astype(np.uint32))
        ctx.pr_init()
        ctx.pr_run()
        for k in range(4):
            rec, have = ops(k)
            ctx.set_params(pull_threshold_div=0 if k == 1 else div)
            ctx.apply_batch(rec)
            a, b = np.array(sorted(have)).T
            M = system(n, a, b)
            want = limit(M, np.zeros(n), np.full(n, (1 - DAMPING) / n))
            r, d = ctx.pr_download()
            assert np.abs(limit(M, r, d) - want).sum() <= tol
            ctx.pr_run()
            r, _ = ctx.pr_download()
            assert np.abs(r - want).sum() <= T / (1 - DAMPING) + tol


@pytest.mark.parametrize("div", [1_000_000, 0], ids=["pull", "push"])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_reseed_of_sources_that_gain_many_edges(gpu, prec, div):
    """Sources of high rank whose degree grows by factors from just below to far above two,
    some losing old edges besides.  The batch itself is held against the exact amendment of
    the state it found: every amended edge takes at most three roundings of a term of its
    source's mass (the contribution, the two additions), so the deltas' error stays under
    eps * 3 * (the mass that the sources sent before and send now + sum |delta|)."""
    rng = np.random.default_rng(17)
    n, k = 6007, 12
    grow = [(1, 5000), (1, 3), (1, 2), (3, 7), (3, 6), (100, 200), (100, 201), (100, 5000), (700, 1401), (2, 300),
            (300, 290), (5, 0)]
    u = [np.arange(100, n)]  # everybody points at one of the sources
    v = [rng.integers(0, k, n - 100)]
    for s, (a, _) in enumerate(grow):
        u.append(np.full(a, s))
        v.append(rng.choice(np.arange(100, n), a, replace=False))
    key = np.unique(np.concatenate(u) * n + np.concatenate(v))
    u, v = key // n, key % n
    off = np.zeros(n + 1, np.uint64)
    off[1:] = np.cumsum(np.bincount(u, minlength=n))
    ops, have = [], set(key.tolist())
    for s, (a, b) in enumerate(grow):
        row = v[u == s]
        assert len(row) == a
        lost = row[: min(a, s % 3 if b > a else a - b)]
        ops += [(1, s, int(t)) for t in lost]
        new = np.setdiff1d(np.arange(100, n), row)
        ops += [(0, s, int(t)) for t in rng.choice(new, max(0, b - a + len(lost)), replace=False)]
        if b > a and len(row) > len(lost):
            ops.append((0, s, int(row[-1])))  # an add of an edge that is there
    rec = np.zeros(len(ops), gpu.UPDATE_DTYPE)
    rec["type"], rec["u"], rec["v"] = np.array(ops).T
    rec = rng.permutation(rec)
    have = (have - {a * n + b for t, a, b in ops if t == 1}) | {a * n + b for t, a, b in ops if t == 0}
    a, b = np.divmod(np.array(sorted(have)), n)
    assert [int((a == s).sum()) for s in range(k)] == [g for _, g in grow]
    M0, M1 = system(n, u, v), system(n, a, b)
    p = gpu.PR_FP64 if prec == "fp64" else gpu.PR_FP32_KAHAN
    eps = 2.0 ** (-53 if prec == "fp64" else -24)
    with gpu.Context(pr_precision=p, termcheck_threshold=1e-6, max_rounds=1000, pull_threshold_div=div) as ctx:
        ctx.upload_csr(off, v.astype(np.uint32))
        ctx.pr_init()
        ctx.pr_run()
        r, d = ctx.pr_download()
        ctx.apply_batch(rec)
        r1, d1 = ctx.pr_download()
    assert np.array_equal(r, r1) and r[0] > 0.02
    sent = DAMPING * r[:k].sum()
    want = d + (M1 - M0) @ r
    assert np.abs(d1 - want).sum() <= eps * 3 * (2 * sent + np.abs(d).sum() + np.abs(want).sum())


@pytest.mark.parametrize("n,m,hot", [(3000, 16383, 0), (3000, 16384, 0), (3000, 16385, 0), (9000, 49157, 0),
                                     (200_000, 100_000, 0), (200_000, 400_000, 0), (5000, 70_001, 8),
                                     (4200, 90_000, 5)])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_binned_layout_at_the_edges_of_its_sort_tiles(gpu, n, m, hot, prec):
    """The binned pull (1 KiB windows) with layouts around whole steps of the ordering
    (8192 edges), a few segments a workgroup and more than its 4096 counters; with `hot`
    sources that reach every vertex, in the hottest range of slots (8), so that a block of
    4096 destinations has a segment of 4096 * hot edges, beyond a chunk (16380)."""
    rng = np.random.default_rng(m)
    key = np.unique((n * rng.random(2 * m) ** 3).astype(np.int64) * n + (n * rng.random(2 * m) ** 2).astype(np.int64))
    key = key[key // n != key % n]
    if hot:
        row = (n * rng.random(m) ** 2).astype(np.int64) % (n - hot) + hot  # the others stay far below n out-edges
        key = np.unique(row * n + rng.integers(0, n, m))
        key = key[key // n != key % n]
        all_of = np.arange(hot * n)
        all_of = all_of[all_of // n != all_of % n]
        key = np.concatenate([all_of, rng.permutation(key)[: m - len(all_of)]])
    key = np.sort(rng.permutation(key)[:m])
    assert len(key) == m
    u, v = key // n, key % n
    off = np.zeros(n + 1, np.uint64)
    off[1:] = np.cumsum(np.bincount(u, minlength=n))
    w = (1.0 - rng.random(m)).astype(np.float32)
    M = system(n, u, v)
    s = np.bincount(u, weights=w.astype(float), minlength=n)
    W = sp.csr_matrix((DAMPING * w.astype(float) / s[u], (v, u)), shape=(n, n))
    T = 1e-11 if prec == "fp64" else 1e-7
    tol = 0.15 * (1e-12 if prec == "fp64" else 1e-5)
    p = gpu.PR_FP64 if prec == "fp64" else gpu.PR_FP32_KAHAN
    x = np.full(n, 1.0 / n, np.float32)
    with gpu.Context(pr_precision=p, termcheck_threshold=T, max_rounds=1000, pull_bin_kib=1) as ctx:
        ctx.upload_csr(off, v.astype(np.uint32), w)
        ctx.pr_init()
        assert ctx.pr_run()["pull_rounds"] > 0
        r, _ = ctx.pr_download()
        ctx.wpr_set_weights(w)
        rw, _ = ctx.wpr_forward(x)
    want = series_limit(M, np.full(n, (1 - DAMPING) / n))
    assert np.abs(r - want).sum() <= T / (1 - DAMPING) + tol
    want = series_limit(W, (1 - DAMPING) * x.astype(float))
    assert np.abs(rw - want).sum() <= T / (1 - DAMPING) + 0.15 * 1e-5  # comes back as FP32
