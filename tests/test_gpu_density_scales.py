"""The density solve's square root and quotient are the correctly rounded ones over the whole range of
lengths: a line of gas from 1e-30 to 1e150 in size, in and out of the range of their short forms
(squares of 1e-250 to 1e250, radii of 1e-120 to 1e120). In one dimension every operation on h and rho
is the oracle's, so they are its bits wherever the same iterations were taken."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def gz():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gizmo_shared_memory_amd import tree
    return tree


@pytest.mark.parametrize("exponent", [-30, -10, 0, 10, 60, 119, 120, 121, 124, 125, 126, 150])
def test_lengths_of_every_scale(gz, oracle, exponent):
    from oracle.bindings import HostParticles
    n = 6000
    rng = np.random.default_rng(7)
    scale = 10.0 ** exponent
    x = rng.uniform(-1.0, 1.0, n)
    x[: n // 3] = 0.4 + 0.03 * rng.normal(size=n // 3)
    h0 = rng.uniform(0.5, 2.0, n) * 6.0 / n * scale
    x *= scale
    case = (x, np.zeros(n), np.zeros(n), rng.uniform(0.5, 1.5, n) / n, np.full(n, 1e-3 * scale))
    tg = np.arange(n, dtype=np.uint32)
    kw = dict(des_ngb=6.0, ngb_tol=0.2, n_dims=1, h_start=h0)
    print(f"[density scales] 1e{exponent}", flush=True)
    P = gz.Particles(*case)
    dev = [v.cpu().numpy() for v in gz.density(gz.build(P), P, tg, **kw)]
    to = oracle.build(HostParticles(*case))
    try:
        ora = oracle.density(to, HostParticles(*case), tg, **kw)
    finally:
        oracle.free(to)
    assert np.array_equal(dev[3], ora[3]) and np.array_equal(dev[2], ora[2])
    assert np.array_equal(dev[0], ora[0]) and np.array_equal(dev[1], ora[1])
    assert np.count_nonzero(ora[3] < 100) > n // 2 and np.isfinite(ora[1]).all()
