"""The exact Hessian product at the edges of its kernels' launch shapes, against the float64 oracle.

The wave tangent and the second-order contractions take the smallest workgroup that holds a
float32 row (128, 256, 512, 1024, 2048 positions): S = 2 L - 1 just below and just above each.
"""

import numpy as np
import pytest
import torch

import kbench_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("leaves", [2, 64, 65, 128, 129, 256, 257, 512, 513, 1024, 1025])
def test_exact_hvp_at_shape_edges_matches_oracle(leaves):
    from kbench import synth
    from kbench.fused import problem_to_captured
    from kbench.newton.hvp import HvpPlan
    from kbench.percall.solve import plan_of, run_forward
    from kbench.runtime import make_static

    problem = synth.build_problem(synth.ProblemConfig(
        leaves, 3, n_nni=1, family_leaves_median=min(12.0, leaves), family_leaves_sigma=0.5, family_leaves_max=40,
        statewise=leaves % 3 != 0, seed=leaves))
    cap = problem_to_captured(problem)
    static = make_static(cap, "cuda")
    theta, cw = cap["inputs"]["theta"].cuda(), cap["inputs"]["col_weights"].cuda()
    prob = O.Problem.from_dict(problem)
    print(f"[hvp edge] S={prob.S}", flush=True)
    _, sv = run_forward(static, theta, cw)
    u = np.random.default_rng(leaves).normal(size=tuple(theta.shape))
    hvp = HvpPlan(plan_of(static), theta, cw, sv, row_classes=leaves % 2 == 0)
    Hu = hvp(torch.as_tensor(u, dtype=theta.dtype).cuda().reshape(-1))
    torch.cuda.synchronize()
    th = np.asarray(problem["inputs"]["theta"], dtype=np.float32).astype(np.float64)
    cw64 = np.asarray(problem["inputs"]["col_weights"], dtype=np.float64)
    _, saved = O.forward(prob, th, cw64)
    _, _, cache = O.build_point_cache(prob, th, cw64, saved)
    ref = O.hvp_exact(prob, th, saved, u, cache).reshape(-1)
    e = np.abs(Hu.double().cpu().numpy() - ref).max() / max(1.0, np.abs(ref).max())
    print(f"  |H u| = {np.abs(ref).max():.4e} rel={e:.3e}")
    assert e <= 1e-3  # the gate of the other Hessian-product parity tests
