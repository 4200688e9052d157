"""The density solve from first guesses and positions at the edges of what it accepts: radii that
are negative or zero, for which the reference's node tests decide what a step finds, and particles
that have since moved beyond any radius, against the oracle."""
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


@pytest.mark.parametrize("x", [1e154, 1e200, np.inf])
def test_live_positions_beyond_any_radius(gz, oracle, x):
    """Particles that have moved so far since the tree's copy of the positions was taken that r / h
    overflows add nothing (W = 0 beyond the kernel), in the wave's kernel and in the rounds. A
    jittered lattice, whose inner particles' corrections (which their infinite moments would switch
    off) do not apply."""
    k = 22
    rng = np.random.default_rng(4)
    g = (np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3) + 0.5 +
         rng.uniform(-0.1, 0.1, (k ** 3, 3))) / k
    case = [np.ascontiguousarray(g[:, d]) for d in range(3)]
    case += [np.full(k ** 3, 1.0 / k ** 3), np.full(k ** 3, 0.01)]
    live = [a.copy() for a in case]
    gone = rng.choice(k ** 3, 40, replace=False)
    live[0][gone] = x
    inner = np.flatnonzero((np.abs(g - 0.5) < 0.2).all(1))
    tg = np.setdiff1d(inner, gone).astype(np.uint32)
    h0 = np.full(tg.shape[0], 0.2)
    print(f"[density guesses] live x={x}", flush=True)
    dev, ora = _both(gz, oracle, case, live, tg, h0, des_ngb=40.0, ngb_tol=0.5)
    _compare(dev, ora)
