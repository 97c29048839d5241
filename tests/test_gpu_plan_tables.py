"""A plan's tables are complete when it is created: a first call that is recorded into a
graph, and so does not run yet, leaves the plan ready for eager calls."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [9, 33])
def test_first_call_recorded_then_eager(M):
    import torch
    from spinifel_amd import engine
    engine.require_gpu()
    print(f"case: M={M}", flush=True)
    rng = np.random.default_rng(M)
    xs = [torch.as_tensor(rng.uniform(-1, 1, 60)).cuda() for _ in range(3)]
    v = torch.as_tensor(rng.standard_normal(60).astype(np.float32)).cuda()
    ac = torch.as_tensor(rng.uniform(size=(M,) * 3).astype(np.float32)).cuda()

    def calls(plan):
        plan.set_model(ac)
        f = plan.execute(*xs, check_domain=False)
        return [f] + [plan.adjoint_points(*xs, values=v, check_domain=False, ordered=o)
                      for o in (False, True)]

    want = [t.clone() for t in calls(engine.NufftPlan(M, 1e-6, 0))]
    plan = engine.NufftPlan(M, 1e-6, 0)
    g = torch.cuda.CUDAGraph()
    # the first calls allocate, which only a relaxed capture lets them
    with torch.cuda.graph(g, capture_error_mode="relaxed"):
        held = calls(plan)
    torch.cuda.synchronize()

    def close(got):
        for a, b in zip(got, want):
            # the atomics' order moves the sums by some 1e-16
            assert float((a - b).norm() / b.norm()) <= 1e-12

    close(calls(plan))
    for _ in range(3):
        for t in held:
            t.zero_()
        g.replay()
        torch.cuda.synchronize()
        close(held)
        close(calls(plan))
