"""FP32 walks of few groups give each group 8, 4 or 2 wavefronts; the results are the bits of one
wavefront's, whatever the group size (lists of several chunks), the stack limit (spilled and
repeated groups) and the target list, and a walk plan's are the same."""
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


# 64-target groups: 8 waves up to 512 expected groups, 4 up to 2,048, 2 up to 5,120, then one
@pytest.mark.parametrize("n", [2, 65, 3000, 24000, 24700, 60000, 99000, 200000, 260000])
@pytest.mark.parametrize("group_size", [64, 200])
def test_group_waves_identical(gz, n, group_size):
    print(f"[group waves] n={n} group_size={group_size}", flush=True)
    P = gz.Particles(*tree_cases.plummer_small(n, seed=61, eps=0.01))
    T = gz.build(P)
    rng = np.random.default_rng(n)
    every = T.device_orderbuf()
    some = torch.as_tensor(np.sort(rng.choice(n, max(1, n // 3), replace=False))
                           .astype(np.uint32).view(np.int32)).cuda().view(torch.uint32)
    for tg in (every, some):
        for theta, limit in ((0.5, 0), (0.2, 512), (0.5, 16)):
            kw = dict(precision="fp32", group_size=group_size)
            one = gz.accel_grouped(T, P, tg, theta, persistent=False, **kw)
            few = gz.accel_grouped(T, P, tg, theta, stack_limit=limit, **kw)
            for u, v in zip(one, few):
                assert torch.equal(u, v), (theta, limit)
    plan = gz.WalkPlan(T, P, some, precision="fp32", group_size=group_size)
    plan.launch(0.5)
    T.ctx.synchronize()
    one = gz.accel_grouped(T, P, some, 0.5, persistent=False, **kw)
    for u, v in zip(one, (plan.ax, plan.ay, plan.az)):
        assert torch.equal(u, v)
