"""Weighted personalized PageRank and its adjoint on the device vs the FP64 oracle
(forward, lambda, both gradients), against central finite differences of the
FP64 device forward, and through the torch.autograd.Function."""
import numpy as np
import pytest

import oracle
from tests.conftest import DAMPING

pytestmark = pytest.mark.gpu


def problem(scale, seed=4, seeds=64):
    g = oracle.Graph.rmat(scale, 16, seed=seed, weights="f32")
    off, col, w = g.csr()
    rng = np.random.default_rng(seed)
    p = np.zeros(g.n, np.float32)
    idx = rng.choice(g.n, seeds, replace=False)
    p[idx] = rng.dirichlet(np.ones(seeds)).astype(np.float32)
    c = rng.standard_normal(g.n).astype(np.float32)
    return g, off, col, w, p, c, rng


# compact=1: both series gather at compact positions by degree (the default only
# above 32 MiB of FP32 state, 8.4M vertices); compact=2 / 3: the binned series
# rounds (1 KiB source windows, the coefficients in layout order) over compact
# positions / vertex ids (the default above 8 MiB of state)
@pytest.mark.parametrize("prec,compact", [("fp64", 0), ("fp32", 0), ("fp64", 1), ("fp32", 1), ("fp64", 2),
                                          ("fp32", 2), ("fp64", 3), ("fp32", 3)])
def test_forward_and_gradients_equal_oracle(gpu, prec, compact):
    g, off, col, w, p, c, _ = problem(14)
    r0, _ = g.wpr_forward(w, p.astype(np.float64), DAMPING)
    lam0, gp0, gw0 = g.wpr_adjoint(w, r0, c.astype(np.float64), DAMPING)
    pp = gpu.PR_FP64 if prec == "fp64" else gpu.PR_FP32_KAHAN
    T = 1e-15 if prec == "fp64" else 1e-9
    kw = {"pull_compact_kib": 1 if compact in (1, 2) else 0}
    if compact >= 2:
        kw["pull_bin_kib"] = 1
    with gpu.Context(pr_precision=pp, termcheck_threshold=T, **kw) as ctx:
        ctx.upload_csr(off, col, w)
        r, st = ctx.wpr_forward(p)
        r64, _ = ctx.wpr_download()
        gp, gw, st2 = ctx.wpr_backward(c)
        _, lam = ctx.wpr_download(adjoint=True)
    if prec == "fp64":
        assert np.abs(r64 - r0).max() < 1e-14
        assert np.abs(lam - lam0).max() < 1e-11 * np.abs(lam0).max()
        assert np.abs(gw - gw0).max() <= 1e-6 * np.abs(gw0).max()  # gw is returned in FP32
    else:
        # FP32 deltas + Kahan FP32 ranks: L1 within 1e-6 of the FP64 fixed point
        assert np.abs(r64 - r0).sum() <= 1e-6
        assert np.abs(lam - lam0).max() <= 1e-4 * np.abs(lam0).max()
        assert np.abs(gw - gw0).max() <= 1e-4 * np.abs(gw0).max()
    assert np.abs(gp - gp0).max() <= 1e-4 * np.abs(gp0).max()
    assert st["rounds"] > 10 and st2["rounds"] > 10


def fd_check(gpu, g, off, col, w, p, c, rng, n_edges, h=1e-3):
    with gpu.Context(pr_precision=gpu.PR_FP32_KAHAN, termcheck_threshold=1e-9) as ctx:
        ctx.upload_csr(off, col, w)
        ctx.wpr_forward(p)
        _, gw, _ = ctx.wpr_backward(c)
    edges = rng.choice(len(w), n_edges, replace=False)
    fds = []
    with gpu.Context(pr_precision=gpu.PR_FP64, termcheck_threshold=1e-15) as ctx:
        ctx.upload_csr(off, col, w)
        for e in edges:
            w1, w2 = w.copy(), w.copy()
            w1[e] += np.float32(h)
            w2[e] -= np.float32(h)
            ctx.wpr_set_weights(w1)
            ctx.wpr_forward(p)
            l1 = c.astype(np.float64) @ ctx.wpr_download()[0]
            ctx.wpr_set_weights(w2)
            ctx.wpr_forward(p)
            l2 = c.astype(np.float64) @ ctx.wpr_download()[0]
            fds.append((l1 - l2) / (np.float64(w1[e]) - np.float64(w2[e])))
    fds = np.array(fds)
    return fds, gw[edges].astype(np.float64)


def test_adjoint_equals_central_differences(gpu):
    """256 random edges, h = 1e-3: the FP32 adjoint gradient against central
    differences of the FP64 forward, within 1e-4 relative."""
    g, off, col, w, p, c, rng = problem(14)
    fd, ga = fd_check(gpu, g, off, col, w, p, c, rng, 256)
    scale = np.abs(fd).max()
    err = np.abs(fd - ga)
    assert np.all(err <= 1e-4 * np.maximum(np.abs(fd), 1e-2 * scale)), (err / np.maximum(np.abs(fd), 1e-30)).max()


def test_weights_update_and_batches(gpu):
    """set_weights re-normalises; an update batch on the graph invalidates the
    forward state and the next forward follows the new graph."""
    g, off, col, w, p, c, rng = problem(12)
    with gpu.Context(pr_precision=gpu.PR_FP64, termcheck_threshold=1e-15) as ctx:
        ctx.upload_csr(off, col, w)
        w2 = (w * rng.uniform(0.5, 1.5, len(w))).astype(np.float32)
        ctx.wpr_set_weights(w2)
        ctx.wpr_forward(p)
        r = ctx.wpr_download()[0]
        assert np.abs(r - g.wpr_forward(w2, p.astype(np.float64), DAMPING)[0]).max() < 1e-14
        ops = g.gen_batch(seed=4, batch_id=0, n_del=100, n_ins=100)
        ops["w_f32"][ops["type"] == 0] = 0.5
        ctx.apply_batch(ops)
        with pytest.raises(gpu.SumincError):
            ctx.wpr_backward(c)  # the forward belongs to the old graph
        g2, _ = oracle.Graph.from_csr(off, col, w2).apply_batch(ops)
        off2, col2, wn = g2.csr()
        ctx.wpr_forward(p)
        r2 = ctx.wpr_download()[0]
        assert np.abs(r2 - g2.wpr_forward(wn, p.astype(np.float64), DAMPING)[0]).max() < 1e-14


def test_wpr_needs_float_weights(gpu):
    g = oracle.Graph.rmat(8, 8, seed=1)
    off, col, _ = g.csr()
    with gpu.Context() as ctx:
        ctx.upload_csr(off, col)
        with pytest.raises(gpu.SumincError) as e:
            ctx.wpr_forward(np.ones(g.n, np.float32) / g.n)
        assert e.value.code == -4


def test_torch_autograd(gpu):
    """The autograd wrapper in a fresh process that imports torch first (torch and
    the library must share one HIP runtime); the case prints OK on success."""
    import subprocess
    import sys
    from pathlib import Path

    case = Path(__file__).with_name("torch_autograd_case.py")
    out = subprocess.run([sys.executable, str(case)], capture_output=True, text=True, timeout=300,
                         cwd=str(case.parent.parent))
    print(out.stdout[-2000:], out.stderr[-2000:])
    if "SKIP" in out.stdout:
        pytest.skip(out.stdout.strip().splitlines()[-1])
    assert out.returncode == 0 and out.stdout.strip().endswith("OK")


@pytest.mark.parametrize("case", ["tile_edges", "long_rows", "sparse_ids", "one_edge"])
@pytest.mark.parametrize("bin_kib", [0, 1], ids=["rows", "binned"])
def test_edge_passes_at_their_edges(gpu, case, bin_kib):
    """Row sums (classes of 32 and 256 edges, 2048-edge chunks), edge tiles (2048 edges,
    rows across them, runs of empty rows on both sides of the search's limit) and layout
    coefficients, through the gradients, against scipy's solve.  FP64 state; gradients
    come back as FP32 (2^-24 of each; 1e-6 of the largest bounds their cancellation)."""
    import scipy.sparse as sp
    import scipy.sparse.linalg as sla

    rng = np.random.default_rng(2)
    if case == "tile_edges":  # row lengths around the classes, the last edge ends a tile
        deg = np.array([0, 1, 8, 9, 31, 32, 33, 64, 255, 256, 257, 0, 0, 300, 7, 2048 - 1253 + 0], int)
        n = 4000
    elif case == "long_rows":
        deg = np.array([2047, 0, 2048, 2049, 4097, 1], int)
        n = 6000
    elif case == "sparse_ids":  # 70,000 and 200,000 empty rows between rows of one tile
        n = 300_000
        deg = np.zeros(270_500, int)
        deg[[0, 1, 70_001, 270_100, 270_499]] = [3, 5, 40, 2, 300]
    else:
        n, deg = 2, np.array([1], int)
    deg = np.concatenate([deg, np.zeros(n - len(deg), int)])
    u = np.repeat(np.arange(n), deg)
    v = np.concatenate([np.sort(rng.choice(n - 1, k, replace=False)) for k in deg if k] or [[]]).astype(np.int64)
    v += v >= u  # no self-loops; still increasing within a row
    off = np.zeros(n + 1, np.uint64)
    off[1:] = np.cumsum(deg)
    if case == "tile_edges":
        assert len(u) % 2048 == 0
    w = (1.0 - rng.random(len(u))).astype(np.float32)
    p = rng.random(n).astype(np.float32) / n
    c = rng.standard_normal(n).astype(np.float32)
    s = np.bincount(u, weights=w.astype(float), minlength=n)
    M = sp.csr_matrix((DAMPING * w.astype(float) / s[u], (v, u)), shape=(n, n))
    I = sp.eye(n, format="csc")
    r = sla.spsolve(I - M.tocsc(), (1 - DAMPING) * p.astype(float))
    lam = sla.spsolve(I - M.T.tocsc(), c.astype(float))
    gw_want = (r / np.where(s > 0, s, 1))[u] * (DAMPING * lam[v] - (M.T @ lam)[u])
    with gpu.Context(pr_precision=gpu.PR_FP64, termcheck_threshold=1e-13, max_rounds=10000,
                     pull_bin_kib=bin_kib or -1) as ctx:
        ctx.upload_csr(off, v.astype(np.uint32), w)
        ctx.wpr_set_weights(w)
        got, _ = ctx.wpr_forward(p)
        gp, gw, _ = ctx.wpr_backward(c)
        dev = [ctx.device_array(x) for x in (p, c, np.zeros(n, np.float32), np.zeros(n, np.float32), np.zeros_like(w))]
        ctx.wpr_forward(dev[0], out=dev[2])
        ctx.wpr_backward(dev[1], grad_p=dev[3], grad_w=dev[4])
        same = [d.download() for d in dev]
        for d in dev:
            d.free()
    assert np.abs(got - r).max() <= 1e-6 * np.abs(r).max()
    assert np.abs(gp - (1 - DAMPING) * lam).max() <= 1e-6 * np.abs(lam).max()
    # (a single edge's gradient is 0: what is left are FP64 roundings of its two terms)
    zero = 1e-14 * (r[u] / s[u]).max() * np.abs(lam).max()
    assert np.abs(gw - gw_want).max() <= 1e-6 * np.abs(gw_want).max() + zero
    # into device memory directly (hub rows add in any order: a last place of FP64 before rounding)
    for x, y in ((same[2], got), (same[3], gp), (same[4], gw)):
        assert np.abs(x - y).max() <= 2e-7 * np.abs(y).max() + zero
    assert np.array_equal(same[0], p) and np.array_equal(same[1], c)


@pytest.mark.parametrize("where", ["device", "host"])
def test_failed_series_leave_the_results_alone(gpu, where):
    """A capped or NaN forward and a capped backward raise and do not write the caller's
    arrays, in device memory as in host memory."""
    g, off, col, w, p, c, _ = problem(10)
    with gpu.Context(termcheck_threshold=1e-12, max_rounds=3) as ctx:
        ctx.upload_csr(off, col, w)
        put = ctx.device_array if where == "device" else (lambda x: x.copy())
        get = (lambda x: x.download()) if where == "device" else (lambda x: x)
        mark = np.full(g.n, -7.0, np.float32)
        r, gp, gw = put(mark), put(mark), put(np.full(len(w), -7.0, np.float32))
        with pytest.raises(gpu.SumincError) as e:
            ctx.wpr_forward(put(p), out=r)
        assert e.value.code == gpu.E_NOT_CONVERGED and (get(r) == -7).all()
        bad = p.copy()
        bad[5] = np.nan
        with pytest.raises(gpu.SumincError) as e:
            ctx.wpr_forward(put(bad), out=r)
        assert e.value.code == gpu.E_NUMERIC and (get(r) == -7).all()
        ctx.set_params(max_rounds=1000)
        ctx.wpr_forward(put(p), out=r)
        assert (get(r) != -7).all()
        ctx.set_params(max_rounds=3)
        with pytest.raises(gpu.SumincError) as e:
            ctx.wpr_backward(put(c), grad_p=gp, grad_w=gw)
        assert e.value.code == gpu.E_NOT_CONVERGED and (get(gp) == -7).all() and (get(gw) == -7).all()
