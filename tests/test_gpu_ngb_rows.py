"""The forward neighbour search around the length of a query's row (64 entries, beyond which a query
is walked again), on both forms of its search nodes (packed from n / 16 queries on), with particles
in and out of their build-time cells, and with buffers that do not hold the lists: every list
against brute force, in slot order."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

N = 6000


@pytest.fixture(scope="module")
def gz():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gizmo_shared_memory_amd import tree
    return tree


@pytest.mark.parametrize("nq", [1, 65, N // 16 - 1, N // 16, 1500])
@pytest.mark.parametrize("aged", [False, True])
def test_lists_around_a_rows_length(gz, nq, aged):
    rng = np.random.default_rng(nq + 7 * aged)
    pos = rng.normal(size=(3, N))
    v = 0.1 * rng.normal(size=(3, N))
    tau = 0.05 if aged else 0.0
    m, soft = np.full(N, 1.0 / N), np.full(N, 0.01)
    T = gz.build(gz.Particles(*pos, m, soft), vel=v)
    now = pos + tau * v
    T.update_sources(gz.Particles(*now, m, soft))
    rank = T.download()["rank"].astype(np.int64)
    c = now[:, rng.choice(N, nq, replace=nq > N)].T
    d2 = ((c[:, None, :] - now.T[None]) ** 2).sum(2)
    want = rng.choice([0, 1, 31, 63, 64, 65, 66, 300], nq)
    srt = np.sort(d2, axis=1)
    r = np.where(want > 0, np.sqrt(0.5 * (srt[np.arange(nq), np.maximum(want - 1, 0)] +
                                          srt[np.arange(nq), want])), 0.0)
    print(f"[ngb rows] nq={nq} aged={aged}", flush=True)
    start, found = gz.ngb_search(T, c, r, tau)
    start, found = start.cpu().numpy(), found.cpu().view(torch.int32).numpy()
    assert start[0] == 0 and start[-1] == found.shape[0]
    for q in range(nq):
        mine = found[start[q]:start[q + 1]]
        every = np.nonzero(d2[q] < r[q] * r[q])[0]
        assert mine.shape[0] == want[q]
        assert np.array_equal(mine, every[np.argsort(rank[every])]), q


@pytest.mark.parametrize("nq,n_long", [(8, 1), (64, 8), (300, 1), (300, 37), (5000, 625),
                                       (5000, 626)])
@pytest.mark.parametrize("aged", [False, True])
def test_few_long_lists(gz, nq, n_long, aged):
    """Up to one query in eight with a list longer than a row: a wave each, as far as one whose
    sphere holds every particle."""
    rng = np.random.default_rng(nq + n_long)
    pos = rng.normal(size=(3, N))
    v = 0.1 * rng.normal(size=(3, N))
    tau = 0.05 if aged else 0.0
    m, soft = np.full(N, 1.0 / N), np.full(N, 0.01)
    T = gz.build(gz.Particles(*pos, m, soft), vel=v)
    now = pos + tau * v
    T.update_sources(gz.Particles(*now, m, soft))
    rank = T.download()["rank"].astype(np.int64)
    c = now[:, rng.choice(N, nq, replace=False)].T
    r = np.zeros(nq)
    longs = np.sort(rng.choice(nq, n_long, replace=False))
    want = rng.choice([65, 128, 129, 1000], n_long)
    want[0] = N
    for q, k in zip(longs, want):
        d = np.sort(((c[q] - now.T) ** 2).sum(1))
        r[q] = np.sqrt(0.5 * (d[k - 1] + (d[k] if k < N else 4 * d[k - 1])))
    print(f"[ngb rows] nq={nq} long={n_long} aged={aged}", flush=True)
    start, found = gz.ngb_search(T, c, r, tau)
    start, found = start.cpu().numpy(), found.cpu().view(torch.int32).numpy()
    assert np.array_equal(np.diff(start)[longs], want) and start[-1] == want.sum()
    for q in longs:
        every = np.nonzero(((c[q] - now.T) ** 2).sum(1) < r[q] * r[q])[0]
        assert np.array_equal(found[start[q]:start[q + 1]], every[np.argsort(rank[every])]), q


def test_buffers_that_do_not_hold_the_lists(gz):
    """The C call with no buffer, one too small, one exactly large enough and one with room for
    long lists: the same total, and the lists where they fit."""
    from gizmo_shared_memory_amd import _lib as L
    rng = np.random.default_rng(3)
    pos = torch.as_tensor(rng.normal(size=(3, N)), device="cuda:0")
    P = gz.Particles(*pos, np.full(N, 1.0 / N), np.full(N, 0.01))
    T = gz.build(P)
    r = torch.full((N,), 0.3, dtype=torch.float64, device="cuda:0")
    start0, found0 = gz.ngb_search(T, pos.t(), r)
    total = int(start0[-1])
    for cap in (0, 1, total - 1, total, total + 5, 70 * N + total):
        start = torch.zeros(N + 1, dtype=torch.int64, device="cuda:0")
        out = torch.full((max(cap, 1) + 1,), -1, dtype=torch.int32, device="cuda:0")
        n = C.c_size_t(0)
        T.ctx.enter()
        assert L.load().gz_tree_ngb_search(
            T.ctx.handle, T.handle, *(a.data_ptr() for a in pos), r.data_ptr(), N, 0.0,
            start.data_ptr(), out.data_ptr() if cap else None, cap, C.byref(n)) == 0
        T.ctx.synchronize()
        assert n.value == total and torch.equal(start, start0)
        if cap >= total:
            assert torch.equal(out[:total], found0.view(torch.int32))
        assert int(out[-1]) == -1
