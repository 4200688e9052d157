"""The density solve where its kernels for the last targets change: 2,048 targets (those of overfull
spheres in the same launch), 131,072 and 393,216 targets in one launch, and 200 and 310 expected
candidates (131 and 204 wanted neighbours in 3D), from guesses far above and below. A target's
result is the same bits in every list, and the oracle's."""
import numpy as np
import pytest

from tests.test_gpu_density import _compare

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

N = 140003


@pytest.fixture(scope="module")
def gz():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gizmo_shared_memory_amd import tree
    return tree


@pytest.fixture(scope="module")
def gas():
    rng = np.random.default_rng(43)
    r = rng.uniform(0.05, 1.0, N) ** 1.2
    u = rng.normal(size=(3, N))
    return r * u / np.sqrt((u * u).sum(0)), r, np.full(N, 1.0 / N), np.full(N, 0.01)


@pytest.mark.parametrize("aged", [False, True])
@pytest.mark.parametrize("des", [32.0, 131.0, 132.0, 203.0, 204.0, 300.0])
def test_every_list_gives_a_targets_result(gz, oracle, gas, des, aged):
    from oracle.bindings import HostParticles
    pos, r, m, soft = gas
    rng = np.random.default_rng(int(des))
    v = 0.05 * rng.normal(size=(3, N))
    tau = 0.02 if aged else 0.0
    now = pos + tau * v
    T = gz.build(gz.Particles(*pos, m, soft), vel=v)
    P = gz.Particles(*now, m, soft)
    T.update_sources(P)
    order = T.device_orderbuf().cpu().view(torch.int32).numpy()
    # about the radius that holds des at the local density, scattered by 40%
    h0 = (des / N * 2.4 * r ** (3.0 - 1.0 / 1.2)) ** (1.0 / 3.0) * 10.0 ** rng.normal(0, 0.15, N)
    kw = dict(des_ngb=des, ngb_tol=1.0, tau=tau)
    print(f"[density limits] des={des} aged={aged}", flush=True)
    every = gz.density(T, P, order, h_start=h0[order], **kw)
    for count in (1, 2048, 2049, 131072, 131073):
        at = np.sort(rng.choice(N, count, replace=False))
        part = gz.density(T, P, order[at], h_start=h0[order[at]], **kw)
        for e, f in zip(every, part):
            assert torch.equal(e[torch.as_tensor(at, device=e.device)], f), count
    at = np.arange(7, N, 701)
    to = oracle.build_vel(HostParticles(*pos, m, soft), v)
    try:
        ora = oracle.density(to, HostParticles(*now, m, soft), order[at].astype(np.uint32),
                             h_start=h0[order[at]], **kw)
    finally:
        oracle.free(to)
    _compare([e[torch.as_tensor(at, device=e.device)] for e in every], ora)


@pytest.mark.parametrize("factor", [1e-3, 30.0])
def test_one_launch_from_far_guesses(gz, oracle, gas, factor):
    """Spheres that start nearly empty, or with a large part of the particles, in the launch that
    takes overfull ones itself and in the one that hands them on."""
    from oracle.bindings import HostParticles
    pos, r, m, soft = gas
    T = gz.build(gz.Particles(*pos, m, soft))
    P = gz.Particles(*pos, m, soft)
    tg = np.arange(3, N, 60, dtype=np.uint32)
    h0 = factor * 0.03 * r[tg]
    print(f"[density limits] factor={factor} targets={tg.shape[0]}", flush=True)
    assert tg.shape[0] > 2048
    kw = dict(des_ngb=32.0, ngb_tol=1.0)
    both = gz.density(T, P, tg, h_start=h0, **kw)
    one = gz.density(T, P, tg[:2000], h_start=h0[:2000], **kw)
    for e, f in zip(both, one):
        assert torch.equal(e[:2000], f)
    to = oracle.build(HostParticles(*pos, m, soft))
    try:
        ora = oracle.density(to, HostParticles(*pos, m, soft), tg[::9], h_start=h0[::9], **kw)
    finally:
        oracle.free(to)
    _compare([e[::9] for e in both], ora)
