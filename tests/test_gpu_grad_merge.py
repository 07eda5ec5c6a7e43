"""The factor cache of the differentiable solve (GPU): a new factor runs on its
plain levels, one that is kept on merged ones, with the same gradients."""
import numpy as np
import pytest

import rchol_amd
from rchol_amd import factor as F
from rchol_amd.solver import OPT_MERGE

pytestmark = pytest.mark.gpu

DIMS = (20, 18, 16)


def tasks_of(prob, w, merge):
    """Sweep tasks of the factor that prob makes of w, with or without merging."""
    Gs, _, _ = F.factor(prob.matrix(w), prob._perm, prob._blocks, prob.order, prob.seed)
    with rchol_amd.Solver() as s:
        s.set_option(OPT_MERGE, merge)
        s.upload_G(Gs, prob.precision)
        st = s.stats()
    return st["fwd_tasks"], st["bwd_tasks"]


@pytest.mark.parametrize("precision", [rchol_amd.FP64, rchol_amd.FP32])
def test_a_factor_that_is_kept_is_merged(precision):
    import torch
    from rchol_amd import autograd as AG
    if rchol_amd.device_count() < 1:
        pytest.skip("no HIP device")
    prob = AG.GridLaplacian(*DIMS, leaves=4, precision=precision, tol=1e-12)
    rng = np.random.default_rng(3)
    weights = [rng.uniform(0.5, 2.0, prob.m) for _ in range(2)]
    b = torch.as_tensor(rng.uniform(-1.0, 1.0, prob.n), device="cuda")

    def forward(wt):
        return ((AG.solve(wt, b, prob) - 1.0) ** 2).sum()

    for w in weights:
        print(f"case kept factor prec={precision}", flush=True)
        plain, merged = tasks_of(prob, w, 0), tasks_of(prob, w, 1)
        assert plain != merged
        wt = torch.as_tensor(w, device="cuda").requires_grad_()
        loss, grads, seen = [], [], []
        for _ in range(6):
            loss.append(forward(wt))
            st = prob.solver_for(wt.detach()).stats() if len(loss) > 5 else prob._solver.stats()
            seen.append((st["fwd_tasks"], st["bwd_tasks"]))
            if len(loss) == 3:
                continue  # its backward runs after the upload of the next pass
            loss[-1].backward()
            grads.append(wt.grad.clone())
            wt.grad = None
        loss[2].backward()
        grads.append(wt.grad.clone())
        # a step of its own (one pass) never pays for the plan
        assert seen == [plain] * AG.MERGE_AT_REUSE + [merged] * (6 - AG.MERGE_AT_REUSE)
        assert prob._factor is None
        for g in grads[1:]:  # both solves to 1e-12
            assert float((g - grads[0]).norm() / grads[0].norm()) <= 1e-9


def test_a_solver_of_other_weights_is_not_reused():
    """solver() between two passes on the same tensor: the second pass has its
    own weights' factor, not the cache's latest."""
    import torch
    from rchol_amd import autograd as AG
    if rchol_amd.device_count() < 1:
        pytest.skip("no HIP device")
    prob = AG.GridLaplacian(*DIMS, leaves=4, precision=rchol_amd.FP64, tol=1e-12)
    rng = np.random.default_rng(5)
    w, other = (rng.uniform(0.5, 2.0, prob.m) for _ in range(2))
    wt = torch.as_tensor(w, device="cuda")
    b = torch.as_tensor(rng.uniform(-1.0, 1.0, prob.n), device="cuda")
    print("case other weights", flush=True)
    x = AG.solve(wt, b, prob)
    prob.solver(10.0 * other)
    y = AG.solve(wt, b, prob)
    assert float((x - y).norm() / x.norm()) <= 1e-9  # both to 1e-12
