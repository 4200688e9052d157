"""FP32 walks of few groups, several wavefronts each, under the relative criterion (aold) and the
learned one: the bits of one wavefront a group, as tests/test_gpu_group_waves.py has them for the
geometric criterion, by a call and by a plan."""
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


@pytest.mark.parametrize("n", [65, 3000, 24700, 99000, 260000])
@pytest.mark.parametrize("learned", [False, True])
def test_group_waves_identical(gz, n, learned):
    from gizmo_shared_memory_amd.learned import load_model
    print(f"[group waves] n={n} learned={learned}", flush=True)
    x, y, z, m, soft = tree_cases.plummer_small(n, seed=62, eps=0.01)
    P = gz.Particles(x, y, z, m, soft)
    T = gz.build(P)
    model = load_model() if learned else None
    rng = np.random.default_rng(n)
    r = np.sqrt(x * x + y * y + z * z)
    aold = 0.0025 * r / (r * r + 1.0) ** 1.5 * 10.0 ** rng.normal(0, 0.2, n)
    every = T.device_orderbuf().cpu().view(torch.int32).numpy()
    some = every[np.sort(rng.choice(n, max(1, n // 5), replace=False))]
    for tg in (every, some):
        kw = dict(precision="fp32", group_size=64, model=model)
        one = gz.accel_grouped(T, P, tg, 0.0, aold=aold[tg], persistent=False, **kw)
        for limit in (0, 512, 16):
            few = gz.accel_grouped(T, P, tg, 0.0, aold=aold[tg], stack_limit=limit, **kw)
            for u, v in zip(one, few):
                assert torch.equal(u, v), limit
        plan = gz.WalkPlan(T, P, tg, **kw)
        plan.launch(0.0, aold=torch.as_tensor(aold[tg], device="cuda"))
        T.ctx.synchronize()
        for u, v in zip(one, (plan.ax, plan.ay, plan.az)):
            assert torch.equal(u, v)
