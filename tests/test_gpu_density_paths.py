"""The density solve's three kernels against the oracle and each other, bit for bit: rounds with a
lane per target (more than 393,216 active targets), a wave per target on collected candidates (the
rest), and a wave per target on the tree (more than 256 candidates). With and without particles
that have left their build-time cells (where the reference's node tests decide), and with particle
types. The device's operations are the reference's in its order; where the two libraries' exp and
log could differ (tolerances of later iterations) only a flipped convergence test would show."""
import numpy as np
import pytest

from tests.test_gpu_density import _compare

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

N = 400003


@pytest.fixture(scope="module")
def gz():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gizmo_shared_memory_amd import tree
    return tree


@pytest.fixture(scope="module")
def gas():
    rng = np.random.default_rng(41)
    r = rng.uniform(0.02, 1.0, N) ** 1.5
    u = rng.normal(size=(3, N))
    pos = r * u / np.sqrt((u * u).sum(0))
    h = 0.9 * (32.0 / N) ** (1.0 / 3.0) * r ** (1.0 / 3.0) * 10.0 ** rng.normal(0, 0.03, N)
    v = 0.2 * rng.normal(size=(3, N))
    ty = (rng.uniform(size=N) < 0.1).astype(np.uint8) * 4
    return pos, np.full(N, 1.0 / N), np.full(N, 0.01), h, v, ty


@pytest.mark.parametrize("aged", [False, True])
@pytest.mark.parametrize("types", [False, True])
def test_rounds_and_waves_match_oracle(gz, oracle, gas, aged, types):
    from oracle.bindings import HostParticles
    pos, m, soft, h, v, ty = gas
    tau = 0.02 if aged else 0.0
    now = pos + tau * v
    kw = dict(des_ngb=32.0, ngb_tol=1.0, tau=tau)
    if types:
        kw["type"] = ty
    print(f"[density paths] aged={aged} types={types}", flush=True)
    T = gz.build(gz.Particles(*pos, m, soft), vel=v)
    P = gz.Particles(*now, m, soft)
    T.update_sources(P)
    order = T.device_orderbuf().cpu().view(torch.int32).numpy()
    assert order.shape[0] > 393216
    every = gz.density(T, P, order, h_start=h[order], **kw)
    at = np.sort(np.random.default_rng(3).choice(N, 700, replace=False))
    at = np.concatenate([at, np.arange(N - 100, N)])
    few = gz.density(T, P, order[at], h_start=h[order[at]], **kw)
    for e, f in zip(every, few):
        assert torch.equal(e[torch.as_tensor(at, device=e.device)], f)
    to = oracle.build_vel(HostParticles(*pos, m, soft), v)
    try:
        ora = oracle.density(to, HostParticles(*now, m, soft), order[at].astype(np.uint32),
                             h_start=h[order[at]], **kw)
    finally:
        oracle.free(to)
    _compare(few, ora)


@pytest.mark.parametrize("des", [8.0, 64.0, 250.0, 400.0])
def test_candidates_beyond_a_waves_registers(gz, oracle, gas, des):
    """250 and more wanted neighbours: the wave's 256 candidates do not hold them."""
    from oracle.bindings import HostParticles
    pos, m, soft, h, _, _ = gas
    n = 30000
    pos, m, soft = pos[:, :n], m[:n], soft[:n]
    at = np.arange(0, n, 97, dtype=np.uint32)
    h0 = h[at] * (N / n * des / 32.0) ** (1.0 / 3.0)
    h0[::5] *= 3.0  # and guesses far above
    print(f"[density paths] des_ngb={des}", flush=True)
    P = gz.Particles(*pos, m, soft)
    T = gz.build(P)
    dev = gz.density(T, P, at, des_ngb=des, ngb_tol=0.5, h_start=h0)
    to = oracle.build(HostParticles(*pos, m, soft))
    try:
        ora = oracle.density(to, HostParticles(*pos, m, soft), at, des_ngb=des, ngb_tol=0.5,
                             h_start=h0)
    finally:
        oracle.free(to)
    _compare(dev, ora)
