"""A build whose arena passes 2^22 nodes, from where on the chunk counts of a level are scanned: from
the start (11.2M particles, a level of 2.1M nodes), and after the arena has grown in the middle of a
build. The trees equal the oracle's bit for bit."""
import types

import numpy as np
import pytest

from tests.treecmp import BIT_FIELDS, assert_same_tree

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gz():
    from gizmo_shared_memory_amd import tree
    return tree


def _same(gz, oracle, case):
    from oracle.bindings import HostParticles
    T = gz.build(gz.Particles(*case))
    d = T.download()
    hp = HostParticles(*case)
    to = oracle.build(hp)
    try:
        o = oracle.tree(to, hp)
        assert np.array_equal(d["skey"], oracle.skeys(to, o.n_live))
        assert np.array_equal(d["orderbuf"], o.orderbuf)
        assert_same_tree(types.SimpleNamespace(**d), o, fields=BIT_FIELDS,
                         what=("device", "oracle"))
    finally:
        oracle.free(to)
    return T


def test_large_level(gz, oracle):
    n = 11186000
    print(f"[build large] n={n}", flush=True)
    rng = np.random.default_rng(3)
    case = (*rng.uniform(-1.0, 1.0, (3, n)), np.full(n, 1.0 / n), np.full(n, 0.01))
    T = _same(gz, oracle, case)
    assert 3 * (2 * n // 16) + 1024 >= 1 << 22 and T.info.arena_grows == 0


def test_arena_grown_past_the_line(gz, oracle):
    """Blocks of 20 particles in two places far closer to each other than to any third: chains of
    one-child nodes to the deepest level."""
    rng = np.random.default_rng(9)
    base = np.repeat(rng.uniform(-1.0, 1.0, (130000, 3)), 20, axis=0)
    xyz = base + 4e-6 * rng.integers(0, 2, base.shape)
    n = xyz.shape[0]
    print(f"[build large] chains, n={n}", flush=True)
    T = _same(gz, oracle, (*(np.ascontiguousarray(xyz[:, d]) for d in range(3)),
                           np.full(n, 1.0 / n), np.full(n, 1e-3)))
    assert T.info.arena_grows >= 1 and T.nnodes > 1 << 20
