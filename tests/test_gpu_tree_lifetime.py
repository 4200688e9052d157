"""Trees and the blocks they leave to their context: a tree freed after its context, and trees freed by
another thread than the one that builds the next ones."""
import threading

import numpy as np
import pytest

from tests import tree_cases

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def gz():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gizmo_shared_memory_amd import tree
    return tree


def _arrays(T):
    return {k: v for k, v in T.download().items() if isinstance(v, np.ndarray)}


def _equal(a, b):
    return all(np.array_equal(a[k], b[k]) for k in a)


def test_tree_freed_after_its_context(gz):
    from gizmo_shared_memory_amd import _lib as L
    P = gz.Particles(*tree_cases.plummer_small(30000, seed=3, eps=0.01))
    want = _arrays(gz.build(P))
    for rounds in range(3):
        print(f"[lifetime] context {rounds}", flush=True)
        ctx = gz.Context(0)
        T, U = gz.build(P, ctx=ctx), gz.build(P, ctx=ctx)
        assert _equal(_arrays(T), want)
        del U  # its blocks are kept by the context ...
        assert L.load().gz_ctx_destroy(ctx.handle) == 0  # ... which gives them back
        del T  # and this tree's go straight back
    assert _equal(_arrays(gz.build(P)), want)


def test_trees_freed_by_another_thread(gz):
    cases = [tree_cases.plummer_small(n, seed=n, eps=0.01) for n in (20000, 21000, 50000)]
    sets = [gz.Particles(*c) for c in cases]
    want = [_arrays(gz.build(P)) for P in sets]
    freed, built, failed = [], threading.Semaphore(0), []

    def free():
        for _ in range(60):
            built.acquire()
            freed.pop(0)  # (the list's reference was the last)
    other = threading.Thread(target=free)
    other.start()
    try:
        for k in range(60):
            i = k % 3
            T = gz.build(sets[i])
            if k % 5 == 0 and not _equal(_arrays(T), want[i]):
                failed.append(k)
            freed.append(T)
            del T
            built.release()
    finally:
        for _ in range(60):
            built.release()
        other.join()
    assert not failed
