"""The per-target walks' two forms, a lane and a wave per target, give the same bits: a list longer
than 24,576 targets takes lanes, shorter ones waves. Both against the oracle, with targets in and
out of tree order, repeated ones, and particles outside the tree."""
import numpy as np
import pytest

from tests import tree_cases

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

WAVE_MAX = 24576


@pytest.fixture(scope="module")
def gz():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gizmo_shared_memory_amd import tree
    return tree


def _cases():
    x, y, z, m, soft = tree_cases.plummer_small(30000, seed=51, eps=0.02)
    yield "plummer", (x, y, z, m, soft)
    m2 = m.copy()
    m2[::9] = 0.0  # outside the tree, still targets
    yield "dead", (x, y, z, m2, soft)
    rng = np.random.default_rng(8)
    k = 30000
    base = np.repeat(rng.uniform(-1, 1, (k // 20, 3)), 20, axis=0)
    p = base + 4e-6 * rng.integers(0, 2, base.shape)  # deep chains and coincident particles
    yield "deep", (*(np.ascontiguousarray(p[:, d]) for d in range(3)), np.full(k, 1.0 / k),
                   np.full(k, 1e-3))


@pytest.mark.parametrize("name", ["plummer", "dead", "deep"])
@pytest.mark.parametrize("theta", [0.0, 0.6])
def test_waves_equal_lanes(gz, oracle, name, theta):
    from oracle.bindings import HostParticles
    case = dict(_cases())[name]
    P = gz.Particles(*case)
    T = gz.build(P)
    rng = np.random.default_rng(2)
    n = P.n
    print(f"[per target] {name} theta={theta}", flush=True)
    tg = rng.permutation(n).astype(np.uint32)
    tg[: n // 50] = tg[n // 2: n // 2 + n // 50]  # repeated targets
    assert n > WAVE_MAX
    aold = rng.uniform(0.001, 0.01, n) if theta == 0.0 else None

    def both(idx):
        a = None if aold is None else aold[idx]
        return (*gz.accel(T, P, tg[idx], theta, aold=a), gz.potential(T, P, tg[idx], theta,
                                                                     aold=a))
    every = both(np.arange(n))
    for count in (1, 2, 63, 64, 65, 1000, WAVE_MAX):
        at = np.sort(rng.choice(n, count, replace=False))
        for e, f in zip(every, both(at)):
            assert torch.equal(e[torch.as_tensor(at, device=e.device)], f), count
    hp = HostParticles(*case)
    to = oracle.build(hp)
    try:
        at = np.arange(0, n, 61)
        a = None if aold is None else aold[at]
        ox, oy, oz = oracle.accel(to, hp, tg[at], theta, 1.0, a)[:3]
        op = oracle.potential(to, hp, tg[at], theta, 1.0, a)
    finally:
        oracle.free(to)
    got = [v.cpu().numpy() for v in both(at)]
    o = np.stack([ox, oy, oz], 1)
    g = np.stack(got[:3], 1)
    assert np.all(np.linalg.norm(g - o, axis=1) <= 1e-12 * np.linalg.norm(o, axis=1) + 1e-300)
    assert np.all(np.abs(got[3] - op) <= 1e-12 * np.abs(op))
