"""The whole-pass driver at the edges of its launch shapes, against the float64 oracle.

Row kernels, E step and backward epilogue take the smallest workgroup that holds the tree
(128, 256, 512, 1024, 1536, 2048, 4096 or 8192 positions): S = 2 L - 1 just below and just above
each of them, with few families so that the oracle stays quick.
"""

import numpy as np
import pytest
import torch

import kbtest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("leaves", [2, 33, 64, 65, 128, 129, 256, 257, 512, 513, 768, 769, 1024, 2049, 4096])
def test_solve_at_shape_edges_matches_oracle(leaves):
    import kbench_oracle as O
    from kbench import synth
    from kbench.fused import FusedSolver, problem_to_captured
    from kbench.runtime import make_static

    weighted, statewise = leaves % 2 == 1, leaves % 3 != 0
    p = synth.build_problem(synth.ProblemConfig(
        leaves, 3, n_nni=2, family_leaves_median=min(9.0, leaves), family_leaves_sigma=0.5, family_leaves_max=30,
        statewise=statewise, seed=leaves))
    cap = problem_to_captured(p)
    static = make_static(cap, "cuda")
    solver = FusedSolver(static, static.solver_options)
    S = solver.S
    cw = (np.random.default_rng(5).normal(0.0, 0.5, size=S) if weighted else np.zeros(S)).astype(np.float32)
    print(f"[shape edge] S={S} C={solver.C} weighted={weighted} statewise={statewise}", flush=True)
    loss, saved, gt, gc = solver.solve(cap["inputs"]["theta"].cuda(), torch.from_numpy(cw).cuda())
    prob = O.Problem.from_dict(p)
    th64 = np.asarray(p["inputs"]["theta"], dtype=np.float32).astype(np.float64)
    ref_loss, ref = O.forward(prob, th64, cw.astype(np.float64))
    ref_gt, ref_gc = O.backward(prob, th64, cw.astype(np.float64), ref)[:2]
    ok, ma, mr = kbtest.compare_inf_safe(saved["pi_wave"].cpu().numpy(), ref["pi_wave"])
    rt, rc = kbtest.norm_rel(gt.cpu().numpy(), ref_gt), kbtest.norm_rel(gc.cpu().numpy(), ref_gc)
    print(f"  pi ok={ok} max_abs={ma:.3e} grad_theta={rt:.3e} grad_col={rc:.3e}")
    # the gates of the other whole-pass parity tests
    assert abs(float(loss) - ref_loss) <= 1e-5 * abs(ref_loss)
    assert ok and (ma <= 2e-4 or mr <= 1e-5)
    assert np.abs(saved["E"].cpu().numpy() - ref["E"]).max() <= 1e-6
    assert rt <= 1e-4 and rc <= 1e-4


@pytest.mark.parametrize("leaves", [65, 513, 1025, 1501, 2049])
def test_backward_of_an_older_forward_matches_its_solve(leaves):
    """Outputs of a forward that is no longer the plan's last: its split terms are gone, and every
    backward kernel recomputes them (the solve's own backward reads the stored ones)."""
    from kbench import synth
    from kbench.fused import FusedSolver, problem_to_captured
    from kbench.runtime import make_static

    cap = problem_to_captured(synth.build_problem(synth.ProblemConfig(
        leaves, 4, n_nni=3, family_leaves_median=12.0, family_leaves_sigma=0.5, family_leaves_max=40,
        statewise=False, seed=leaves)))
    static = make_static(cap, "cuda")
    solver = FusedSolver(static, static.solver_options)
    theta = cap["inputs"]["theta"].cuda()
    cw = torch.from_numpy(np.random.default_rng(7).normal(0.0, 0.5, size=solver.S).astype(np.float32)).cuda()
    _, saved, gt, gc = solver.solve(theta, cw)
    solver.run_forward(theta - 0.5, cw)
    gt2, gc2 = solver.run_backward(theta, cw, saved)
    print(f"[older forward] S={solver.S}", flush=True)
    # the split terms differ by float32 rounding only (exp2 / log2 of the two kernels)
    assert kbtest.norm_rel(gt2.cpu().numpy(), gt.cpu().numpy()) <= 1e-5
    assert kbtest.norm_rel(gc2.cpu().numpy(), gc.cpu().numpy()) <= 1e-5
