"""Neighbour lists that a lane gives up (64 entries per query of its wave and more) and that a wave of
its own counts and fills, at the numbers of queries where a wave holds one, two, four and 64 of
them, with rows and without, fresh and aged trees: every list against brute force, in slot order."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

N = 9000


@pytest.fixture(scope="module")
def gz():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gizmo_shared_memory_amd import tree
    return tree


# 256 CUs hold 4,096 waves: up to 4,096 queries one to a wave, two to 8,192, four to 16,384, 64 from
# 262,081 on
@pytest.mark.parametrize("nq,n_long", [(4096, 5), (4097, 1), (8192, 700), (8193, 1), (12000, 9000),
                                       (262081, 3)])
@pytest.mark.parametrize("aged", [False, True])
def test_lists_given_up_by_lanes(gz, nq, n_long, aged):
    from gizmo_shared_memory_amd import _lib as L
    rng = np.random.default_rng(nq + n_long)
    pos = rng.normal(size=(3, N))
    v = 0.1 * rng.normal(size=(3, N))
    tau = 0.05 if aged else 0.0
    T = gz.build(gz.Particles(*pos, np.full(N, 1.0 / N), np.full(N, 0.01)), vel=v)
    now = pos + tau * v
    T.update_sources(gz.Particles(*now, np.full(N, 1.0 / N), np.full(N, 0.01)))
    qpw = 64
    while qpw > 1 and -(-nq // qpw) < 4096:
        qpw //= 2
    of = rng.integers(0, N, nq)
    c = torch.as_tensor(np.ascontiguousarray(now[:, of]), device="cuda")
    p = torch.as_tensor(now, device="cuda")
    rank = torch.as_tensor(T.download()["rank"].astype(np.int64), device="cuda")
    longs = np.sort(rng.choice(nq, n_long, replace=False))
    most = [64 * qpw - 1, 64 * qpw, 64 * qpw + 1, 2 * 64 * qpw + 3, N]
    want = torch.zeros(nq, dtype=torch.int64, device="cuda")
    r = torch.zeros(nq, dtype=torch.float64, device="cuda")
    for lo in range(0, n_long, 500):
        at = torch.as_tensor(longs[lo:lo + 500], device="cuda")
        d2 = sum((c[k][at][:, None] - p[k][None]) ** 2 for k in range(3))
        srt = torch.sort(d2, 1).values
        k = torch.as_tensor([min(m, N) for m in rng.permutation(most * 101)[:at.shape[0]]],
                            device="cuda")
        if n_long > 100:
            k = k.clamp(max=129)  # (their sum is to fit one call)
        i = torch.arange(at.shape[0], device="cuda")
        far = torch.where(k < N, srt[i, k.clamp(max=N - 1)], 2.0 * srt[i, k - 1])
        r[at] = torch.sqrt(0.5 * (srt[i, k - 1] + far))
        want[at] = k
    total = int(want.sum())
    print(f"[ngb long] nq={nq} qpw={qpw} long={n_long} aged={aged} total={total}", flush=True)
    for cap in (total, 70 * nq + total):  # rows, no rows
        start = torch.zeros(nq + 1, dtype=torch.int64, device="cuda")
        found = torch.full((cap + 1,), -1, dtype=torch.int32, device="cuda")
        n = C.c_size_t(0)
        T.ctx.enter()
        L.check(L.load().gz_tree_ngb_search(
            T.ctx.handle, T.handle, *(a.data_ptr() for a in c), r.data_ptr(), nq, tau,
            start.data_ptr(), found.data_ptr(), cap, C.byref(n)), "gz_tree_ngb_search")
        T.ctx.synchronize()
        assert n.value == total and torch.equal(start[1:] - start[:-1], want)
        assert bool((found[total:] == -1).all())
        for q in longs[:: max(1, n_long // 300)]:
            d2 = sum((c[k][q] - p[k]) ** 2 for k in range(3))
            every = torch.nonzero(d2 < r[q] * r[q])[:, 0]
            every = every[torch.argsort(rank[every])]
            assert torch.equal(found[start[q]:start[q + 1]].long(), every), q
