"""Results in pageable host memory, at the edges of the pinned chunks they cross in
(2 MiB: 262,144 doubles, 524,288 words; 16 slots; threads from 4 MiB on), in several
threads at once, and in device memory."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def state(ctx, n, seed):
    rng = np.random.default_rng(seed)
    r, d = rng.random(n), rng.standard_normal(n)
    ctx.upload_csr(np.zeros(n + 1, np.uint64), np.zeros(0, np.uint32))
    ctx.pr_upload(r, d)
    return r, d


@pytest.mark.parametrize("n", [1, 1000, 131071, 262143, 262144, 262145, 16 * 262144 + 3, 40 * 262144 - 1])
def test_ranks_arrive_whole(gpu, n):
    with gpu.Context(pr_precision=gpu.PR_FP64) as ctx:
        r, d = state(ctx, n, n)
        for _ in range(2):
            gr, gd = ctx.pr_download()
            assert np.array_equal(gr, r) and np.array_equal(gd, d)
        only = np.zeros(n)
        ctx._check(ctx._lib.suminc_pr_download(ctx._h, None, only.ctypes.data_as(C.c_void_p)))
        assert np.array_equal(only, d)
        dev = ctx.device_array(np.zeros(n))  # device memory takes the other way
        ctx._check(ctx._lib.suminc_pr_download(ctx._h, dev.ptr, None))
        assert np.array_equal(dev.download(), r)
        dev.free()


@pytest.mark.parametrize("n", [2, 524287, 524289, 17 * 524288 + 1])
def test_distances_and_parents_arrive_whole(gpu, n):
    rng = np.random.default_rng(n)
    up = (rng.random(n - 1) * np.arange(1, n)).astype(np.int64)  # a tree: up[v - 1] < v
    order = np.argsort(up, kind="stable")
    off = np.zeros(n + 1, np.uint64)
    off[1:] = np.cumsum(np.bincount(up, minlength=n))
    depth = np.full(n, -1, np.int64)
    depth[0] = 0
    while (depth < 0).any():
        known = depth[up] >= 0
        depth[1:][known] = depth[up[known]] + 1
    with gpu.Context() as ctx:
        ctx.upload_csr(off, (order + 1).astype(np.uint32))
        ctx.traversal_init(gpu.APP_BFS, 0)
        ctx.sssp_run()
        dist, par = ctx.sssp_download()
    assert np.array_equal(dist, depth)
    assert np.array_equal(par[1:], up)


@pytest.mark.parametrize("threads", [4, 12])
def test_threads_read_back_at_once(gpu, threads):
    """Each with pinned slots of its own; beyond eight, some the runtime's way."""
    bad = []

    def one(seed):
        n = (600_000 if threads == 4 else 300_000) + seed
        with gpu.Context(pr_precision=gpu.PR_FP64) as ctx:
            r, d = state(ctx, n, seed)
            for _ in range(5):
                gr, gd = ctx.pr_download()
                if not (np.array_equal(gr, r) and np.array_equal(gd, d)):
                    bad.append(seed)

    ts = [threading.Thread(target=one, args=(k,)) for k in range(threads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
