"""The device build at the sizes where its kernels change form: the sort's tiles (4,096 particles
from 2^20 on, 2,048 below) and its direct scatter (to 128 tiles), the packed gather (from 2^19),
particle sets with dead members, levels enqueued in several batches, and an arena that has to grow
in the middle of a level. Every tree must equal the oracle's bit for bit."""
import types

import numpy as np
import pytest

from tests.treecmp import BIT_FIELDS, assert_same_tree

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gz():
    from gizmo_shared_memory_amd import tree
    return tree


@pytest.fixture(scope="module")
def oracle():
    from oracle.bindings import Oracle
    return Oracle()


def _particles(n, dead, seed):
    """Half of the particles uniform in a box, half in clumps of one to 40 within 1e-4 of it, a
    few of them on top of each other; every dead-th one massless."""
    rng = np.random.default_rng(seed)
    k = n // 2
    xyz = rng.uniform(-1.0, 1.0, (n, 3))
    centre = np.repeat(rng.uniform(-1.0, 1.0, (max(k // 20, 1), 3)), 20, axis=0)[:k]
    xyz[: centre.shape[0]] = centre + 1e-4 * rng.uniform(-1.0, 1.0, centre.shape)
    xyz[: k // 16] = xyz[k // 16: 2 * (k // 16)]
    perm = rng.permutation(n)
    m = rng.uniform(0.5, 1.5, n) / n
    if dead:
        m[::dead] = 0.0
    x, y, z = (np.ascontiguousarray(xyz[perm, d]) for d in range(3))
    return x, y, z, m, rng.uniform(0.0, 0.01, n)


def _check(gz, oracle, case):
    from oracle.bindings import HostParticles
    P = gz.Particles(*case)
    T = gz.build(P)
    d = T.download()
    hp = HostParticles(*case)
    to = oracle.build(hp)
    try:
        o = oracle.tree(to, hp)
        assert d["n_live"] == o.n_live
        assert np.array_equal(d["skey"], oracle.skeys(to, o.n_live))
        assert np.array_equal(d["orderbuf"], o.orderbuf)
        assert np.array_equal(d["rank"], o.rank)
        assert_same_tree(types.SimpleNamespace(**d), o, fields=BIT_FIELDS,
                         what=("device", "oracle"))
        assert T.info.nleaves == int((d["first"] < 0).sum())
    finally:
        oracle.free(to)
    return P, T, d


@pytest.mark.parametrize("n,dead", [(16385, 0), (262143, 0), (262145, 3), (524287, 0),
                                    (524289, 7), (1048575, 0), (1048577, 0), (1048583, 2)])
def test_build_matches_oracle_at_kernel_edges(gz, oracle, n, dead):
    print(f"[build sizes] n={n} dead={dead}", flush=True)
    P, T, d = _check(gz, oracle, _particles(n, dead, 5))
    # the sources read again from the particles are what the build gathered
    a = gz.accel(T, P, d["orderbuf"][:257], 0.7)
    T.update_sources()
    b = gz.accel(T, P, d["orderbuf"][:257], 0.7)
    for u, v in zip(a, b):
        assert bool((u == v).all())


def test_arena_grows_between_levels(gz, oracle):
    """Pairs of particles far closer to each other than to any third: chains of one-child nodes
    down to the deepest level, many more nodes than the arena first holds."""
    rng = np.random.default_rng(9)
    k = 4000
    base = np.repeat(rng.uniform(-1.0, 1.0, (k // 20, 3)), 20, axis=0)
    xyz = base + 4e-6 * rng.integers(0, 2, base.shape)
    m = np.full(k, 1.0 / k)
    case = (*(np.ascontiguousarray(xyz[:, d]) for d in range(3)), m, np.full(k, 1e-3))
    P, T, d = _check(gz, oracle, case)
    assert T.info.arena_grows >= 1 and T.info.depth >= 18
    with pytest.raises(Exception, match="max_nodes"):
        gz.build(P, max_nodes=200)


def test_freed_blocks_serve_other_trees(gz, oracle):
    """Trees of different sizes built and freed in turn reuse each other's device blocks, with and
    without velocities, and while another tree is alive."""
    keep, kt, _ = _check(gz, oracle, _particles(30000, 0, 6))
    want = gz.accel(kt, keep, np.arange(200), 0.7)
    for n, dead in ((30001, 0), (29000, 5), (60000, 0), (30001, 2)):
        case = _particles(n, dead, n)
        _check(gz, oracle, case)
        P = gz.Particles(*case)
        T = gz.build(P, vel=case[:3])
        T.refresh_walk_nodes(0.0)
        got = T.download()
        ref = gz.build(P).download()
        for f in ("mass", "cx", "cy", "cz", "soft", "first", "plo", "leaf_of", "rank"):
            assert np.array_equal(got[f], ref[f]), f
        del T
    for u, v in zip(want, gz.accel(kt, keep, np.arange(200), 0.7)):
        assert bool((u == v).all())
