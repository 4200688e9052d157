"""The density solve from first guesses and positions at the edges of what it accepts: radii that
are negative or zero, for which the reference's node tests decide what a step finds, against the
oracle."""
import numpy as np
import pytest

from tests.test_gpu_density import _compare
from tests.test_oracle_density import _gas

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def gz():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gizmo_shared_memory_amd import tree
    return tree


def _both(gz, oracle, case, live, tg, h0, **kw):
    """The device's and the oracle's solve on the tree of case, the particles now at live."""
    from oracle.bindings import HostParticles
    T = gz.build(gz.Particles(*case))
    dev = gz.density(T, gz.Particles(*live), tg, h_start=h0, **kw)
    to = oracle.build(HostParticles(*case))
    try:
        return dev, oracle.density(to, HostParticles(*live), tg, h_start=h0, **kw)
    finally:
        oracle.free(to)


@pytest.mark.parametrize("dims", [1, 2, 3])
@pytest.mark.parametrize("scale", [1.0, 1e-3])
def test_negative_and_zero_guesses(gz, oracle, dims, scale):
    """A step from a negative radius moves to one of larger size: what it finds there is not what
    the step before it found."""
    case = _gas(8000, dims, seed=3)
    rng = np.random.default_rng(1)
    tg = np.arange(0, 8000, 5, dtype=np.uint32)
    h0 = scale * rng.uniform(0.02, 0.2, tg.shape[0])
    h0[::2] *= -1.0
    h0[::7] = 0.0
    print(f"[density guesses] dims={dims} scale={scale}", flush=True)
    dev, ora = _both(gz, oracle, case, case, tg, h0, des_ngb={3: 32.0, 2: 20.0, 1: 6.0}[dims],
                     ngb_tol=1.0, n_dims=dims)
    assert np.count_nonzero(ora[3] == 100) > tg.shape[0] // 2  # they do not leave the sign
    _compare(dev, ora)
