"""The per-call E step, its fixed point and its VJP at the edges of their launch shapes, against the oracle.

Item rows whose parameters all lie in [-400, 200] (log2) run in linear float64, any other row in
log space: one row of each launch has a probability of 0 and one a rate of 2^-600.
"""

import numpy as np
import pytest
import torch

import kbench_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("leaves", [2, 64, 65, 128, 129, 256, 257, 512, 513, 1024, 1025, 2049])
@pytest.mark.parametrize("weighted", [False, True])
def test_e_step_rows_match_oracle(leaves, weighted):
    from kbench import synth
    from kbench.core.kernels.e_step import e_fixed_point_triton, e_step_triton_autograd

    rng = np.random.default_rng(leaves)
    tree = synth.yule_tree(leaves, rng)
    h = synth.state_helpers_from_tree(tree)
    S, G = tree.S, 4
    logits = rng.uniform(-3.0, -1.0, (G, S, 3))
    r = O.log2_softmax(np.concatenate([np.zeros((G, S, 1)), logits], axis=-1))
    pS, pD, pL, pT = (r[..., k].copy() for k in range(4))
    pL[2, : leaves // 2] = -np.inf      # leaves that cannot go extinct by loss
    pD[3, S - 1] = -600.0
    col = np.log2(rng.dirichlet(np.full(S, 20.0))) if weighted else np.full(S, -np.log2(S))
    otree = O.Tree.from_helpers(h)
    norm = O.col_valid_log_normalizer(col, otree) if weighted else np.asarray(h["unnorm_row_max"])
    mt = pT + norm
    E0 = np.full((G, S), -1.0)
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda")
    topo = [torch.as_tensor(np.asarray(h[k])).cuda() for k in ("node_parent", "node_child1", "node_child2")]
    topo.append(int(h["max_ancestor_depth"]))
    print(f"[e step] S={S} weighted={weighted}", flush=True)
    params = [t(x) for x in (pS, pD, pL, mt)]
    got = e_fixed_point_triton(t(E0), *params, t(col), *topo, max_iter=500, tol=1e-10, use_col_weights=weighted)
    with np.errstate(all="ignore"):
        want = [np.empty((G, S)) for _ in range(4)]
        for g in range(G):  # rows stop on their own
            row = lambda a: a[g:g + 1]
            for o, x in zip(want, O.e_fixed_point(row(E0), row(pS), row(pD), row(pL), row(mt), col, otree, weighted,
                                                  500, 1e-10)):
                o[g] = x[0]
    # an iterate at the stopping line may take one more step: 1e-10; the others' sum is a difference
    # of prefix sums of S values (float64)
    for name, a, b in zip(("E", "E_s1", "E_s2", "Ebar"), got, want):
        a = a.cpu().numpy()
        assert np.array_equal(np.isfinite(a), np.isfinite(b)), name
        f = np.isfinite(b)
        assert np.abs(a[f] - b[f]).max(initial=0.0) <= 1e-9, name
    # one step and its VJP at that point
    E = want[0]
    cot = [rng.normal(size=(G, S)) for _ in range(4)]
    for c, o in zip(cot, O.e_step(E, pS, pD, pL, mt, col, otree, weighted)):
        c[~np.isfinite(o)] = 0.0  # (an output of -inf has no cotangent)
    leaves_ = [x.requires_grad_(True) for x in (t(E), *(p.clone() for p in params), t(col))]
    out = e_step_triton_autograd(*leaves_, *topo, use_col_weights=weighted)
    with np.errstate(all="ignore"):
        ref = O.e_step(E, pS, pD, pL, mt, col, otree, weighted)
        ref_g = O.e_step_vjp(E, pS, pD, pL, mt, col, otree, weighted, *cot)
    for a, b in zip(out, ref):
        a = a.detach().cpu().numpy()
        assert np.array_equal(np.isfinite(a), np.isfinite(b))
        f = np.isfinite(b)
        assert np.abs(a[f] - b[f]).max(initial=0.0) <= 1e-10
    grads = torch.autograd.grad(out, leaves_, grad_outputs=[t(c) for c in cot])
    for name, a, b in zip(("E", "pS", "pD", "pL", "mt", "col"), grads, ref_g):
        assert np.abs(a.cpu().numpy() - b).max() <= 1e-10 * max(1.0, np.abs(b).max()), name


@pytest.mark.parametrize("leaves", [2, 64, 300, 1024, 2049])
def test_large_values_stay_finite(leaves):
    """Steps whose products pass 2^1024 (unnormalised rates), and a fixed point that grows past it: log space."""
    from kbench import synth
    from kbench.core.kernels.e_step import e_fixed_point_triton, e_step_triton_autograd

    rng = np.random.default_rng(leaves)
    h = synth.state_helpers_from_tree(synth.yule_tree(leaves, rng))
    S, G = 2 * leaves - 1, 3
    otree = O.Tree.from_helpers(h)
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda")
    topo = [torch.as_tensor(np.asarray(h[k])).cuda() for k in ("node_parent", "node_child1", "node_child2")]
    topo.append(int(h["max_ancestor_depth"]))
    print(f"[large e] S={S}", flush=True)
    for weighted in (False, True):
        col = rng.uniform(190.0, 199.0, S) if weighted else np.full(S, -np.log2(S))
        E, pS, pD, pL, mt = (rng.uniform(-3.0, -1.0, (G, S)) for _ in range(5))
        E[1], pS[1], pD[1], mt[1] = (rng.uniform(340.0, 399.0, S) for _ in range(4))
        E[2] = 199.0
        mt[2] = pD[2] = 190.0
        out = e_step_triton_autograd(*(t(x) for x in (E, pS, pD, pL, mt, col)), *topo, use_col_weights=weighted)
        with np.errstate(all="ignore"):
            ref = O.e_step(E, pS, pD, pL, mt, col, otree, weighted)
        for a, b in zip(out, ref):
            a = a.cpu().numpy()
            assert np.array_equal(np.isfinite(a), np.isfinite(b))
            f = np.isfinite(b)
            assert np.abs(a[f] - b[f]).max(initial=0.0) <= 1e-10 * max(1.0, np.abs(b[f]).max(initial=0.0))
        # no transfers to speak of and every other rate 1: the exponents double with every step
        one = np.zeros((G, S))
        got = e_fixed_point_triton(t(one + 150.0), *(t(one + x) for x in (0.0, 0.0, 0.0, -390.0)), t(col), *topo,
                                   max_iter=3, tol=1e-8, use_col_weights=weighted)
        with np.errstate(all="ignore"):
            want = O.e_fixed_point(one + 150.0, one, one, one, one - 390.0, col, otree, weighted, 3, 1e-8)
        assert np.isfinite(want[0]).all() and want[0].max() > 1100.0
        for a, b in zip(got, want):
            a = a.cpu().numpy()
            assert np.array_equal(np.isfinite(a), np.isfinite(b))
            f = np.isfinite(b)
            assert np.abs(a[f] - b[f]).max(initial=0.0) <= 1e-9 * np.abs(b[f]).max(initial=1.0)


@pytest.mark.parametrize("leaves", [2, 65, 300, 1024, 2049])
@pytest.mark.parametrize("mode", [0, 1])
def test_e_out_may_be_e(leaves, mode):
    """The entry point called in place gives the bits of a call with a row block of its own, in both forms."""
    from kbench import synth
    from kbench.core.kernels import _hip as H

    rng = np.random.default_rng(leaves)
    h = synth.state_helpers_from_tree(synth.yule_tree(leaves, rng))
    S, G = 2 * leaves - 1, 3
    print(f"[in place] S={S} mode={mode}", flush=True)
    tree = H.tree_from_parent(*(torch.as_tensor(np.asarray(h[k])).cuda()
                                for k in ("node_parent", "node_child1", "node_child2")))
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float32, device="cuda")
    par = [rng.uniform(-5.0, -2.0, (G, S)) for _ in range(3)] + [rng.uniform(-16.0, -12.0, (G, S))]
    par[1][1] = -np.inf  # a row in log space
    par, col = [t(x) for x in par], t(np.full(S, -np.log2(S)))
    E = t(rng.uniform(-3.0, -1.0, (G, S)))
    res = []
    for in_place in (False, True):
        src = E.clone()
        outs = [src if in_place else torch.empty_like(E)] + [torch.empty_like(E) for _ in range(3)]
        diff = torch.full((G,), -7.0, device="cuda")
        io = H.KbEStepIO(dtype=H.KB_F32, G=G, mode=mode, use_col_weights=0, max_iter=20, tol=1e-6, E=H.ptr(src),
                         log_pS=H.ptr(par[0]), log_pD=H.ptr(par[1]), log_pL=H.ptr(par[2]), max_coupling=H.ptr(par[3]),
                         col_log_probs=H.ptr(col), E_out=H.ptr(outs[0]), E_s1=H.ptr(outs[1]), E_s2=H.ptr(outs[2]),
                         Ebar=H.ptr(outs[3]), max_diff=H.ptr(diff), n_iter=None)
        H.check(H.lib().kb_estep(tree.handle, io, H.stream(E.device)))
        torch.cuda.synchronize()
        res.append([x.cpu() for x in outs] + [diff.cpu()])
    for a, b in zip(*res):
        assert torch.equal(a, b)
