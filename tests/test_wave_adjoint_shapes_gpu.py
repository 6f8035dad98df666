"""The wave adjoint's kernels at the edges of their launch shapes, against the float64 oracle.

``wave_backward_uniform_fused``, ``dts_cross_backward_accum_fused`` and
``uniform_cross_pibar_vjp_tree_from_ud_fused`` take the smallest workgroup that holds a row;
the added rows go to children named by one split, by several and by both sides of one.
"""

import numpy as np
import pytest
import torch

import kbench_oracle as O

pytestmark = pytest.mark.gpu

W, N_CHILD = 4, 9  # parent rows 9 .. 12; children 0 .. 8
SL, SR = np.array([0, 1, 3, 3, 4, 6]), np.array([1, 2, 2, 5, 4, 7])
RED = np.array([0, 0, 1, 2, 2, 3])


@pytest.mark.parametrize("leaves,kind", [(n, k) for n in (2, 64, 65, 128, 129, 256, 257, 512, 513, 1024, 1025, 2049)
                                         for k in ("float32", "float64")])
def test_wave_adjoint_at_shape_edges_matches_oracle(leaves, kind):
    from kbench import synth
    from kbench.core.kernels import wave_backward as wb

    dt, tdt = (np.float32, torch.float32) if kind == "float32" else (np.float64, torch.float64)
    weighted = leaves % 2 == 1
    rng = np.random.default_rng(leaves)
    h = synth.state_helpers_from_tree(synth.yule_tree(leaves, rng))
    tree = O.Tree.from_helpers(h)
    S, C = tree.S, N_CHILD + W
    print(f"[wave adjoint] S={S} {kind} weighted={weighted}", flush=True)
    rnd = lambda a: np.asarray(a, dtype=np.float64).astype(dt).astype(np.float64)
    par = {k: rnd(rng.uniform(-4.0, -1.0, (1, S))) for k in ("pS", "pD", "E", "Ebar", "SL1", "SL2", "DL")}
    mt = rnd(rng.uniform(-1.0, 0.0, (1, S)) - np.log2(S))
    col = rnd(rng.normal(0.0, 0.5, S)) if weighted else np.zeros(S)
    item = np.zeros(C, dtype=np.int64)
    lsp = rnd(np.log2(rng.uniform(0.2, 0.8, SL.size)))
    meta = dict(sl=SL, sr=SR, reduce_idx=RED, log_split_probs=lsp)
    Pi = rng.uniform(-12.0, -2.0, (C, S))
    Pi[2, rng.random(S) < 0.3] = -np.inf
    Pi = rnd(Pi)
    Pb, rmax = np.zeros((C, S)), np.zeros(C)
    with np.errstate(all="ignore"):
        b = O._pibar_from_pi(Pi[:N_CHILD], col, np.repeat(mt, N_CHILD, 0), tree, weighted)
        Pb[:N_CHILD], rmax[:N_CHILD] = rnd(b[0]), rnd(b[1])
        dts = rnd(O.dts_forward(Pi, Pb, meta, W, par["pD"], par["pS"], item, N_CHILD, tree))
        Pi[N_CHILD:] = rnd(dts + 0.25)
        b = O._pibar_from_pi(Pi[N_CHILD:], col, np.repeat(mt, W, 0), tree, weighted)
        Pb[N_CHILD:], rmax[N_CHILD:] = rnd(b[0]), rnd(b[1])
    rhs = -np.abs(rng.normal(size=(W, S)))
    rhs[1] = 0.0  # an inactive row
    rhs = rnd(rhs)
    act = np.array([True, False, True, True])
    rows = np.arange(N_CHILD, C)
    consts = O.WaveConsts(mt=mt, DL=par["DL"], Ebar=par["Ebar"], E=par["E"], SL1=par["SL1"], SL2=par["SL2"],
                          leaf_logp=par["pS"], col=col, use_col_weights=weighted)
    # sums of up to S terms in the call's type: half an ulp each at the most, and a few ulp of the exponentials
    tol = 1e-9 if dt is np.float64 else (S + 64) * 2.0**-24

    def close(got, ref, name):
        got, ref = got.detach().double().cpu().numpy(), np.asarray(ref)
        assert np.isfinite(got).all(), name
        assert np.abs(got - ref).max() <= tol * max(1.0, np.abs(ref).max()), name

    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=tdt, device="cuda")
    ints = lambda a: torch.as_tensor(np.asarray(a), dtype=torch.int64, device="cuda")
    hd = {k: torch.as_tensor(np.asarray(v)).cuda() if isinstance(v, np.ndarray) else v for k, v in h.items()}
    levels = {k: hd[k] for k in ("compact_level_ptr", "compact_level_parents", "compact_level_child1",
                                 "compact_level_child2")}
    actd = torch.as_tensor(act).cuda()
    d = lambda k: t(par[k])
    ref = O.wave_backward_uniform(Pi[rows], Pb[rows], rmax[rows], rhs, item[rows], consts, tree, 4, active=act, dts_r=dts)
    gcol = torch.zeros((S,), dtype=tdt, device="cuda")
    got = wb.wave_backward_uniform_fused(
        t(Pi), t(Pb), N_CHILD, W, S, t(dts), t(rhs), t(mt), d("DL"), d("Ebar"), d("E"), d("SL1"), d("SL2"), t(col),
        hd["node_child1"], hd["node_child2"], None, neumann_terms=4, leaf_state_idx=ints(np.zeros(C)), leaf_logp=d("pS"),
        has_leaf_term=False, active_mask=actd, node_parent=hd["node_parent"],
        max_ancestor_depth=int(h["max_ancestor_depth"]), pibar_row_max=t(rmax), item_idx=ints(item),
        item_indexed_consts=True, grad_col_log_probs=gcol, use_col_weights=weighted, **levels)
    torch.cuda.synchronize()
    for k, (g, r) in enumerate(zip([*got, gcol], ref)):
        if g is not None:
            close(g[actd] if k == 0 else g, r[act] if k == 0 else r, f"wave backward output {k}")

    v = np.where(act[:, None], got[0].double().cpu().numpy(), 0.0)
    with np.errstate(all="ignore"):
        ref = O.dts_cross_backward(Pi, Pb, rmax, v, N_CHILD, meta, par["pD"], par["pS"], mt, item, tree, act, col, weighted)
    acc = torch.zeros((C, S), dtype=tdt, device="cuda")
    g_pD, g_pS, g_mt = (torch.zeros((1, S), dtype=tdt, device="cuda") for _ in range(3))
    ud, A, side, _, _ = wb.dts_cross_backward_accum_fused(
        t(Pi), t(Pb), t(v), N_CHILD, ints(SL), ints(SR), ints(RED), t(lsp), d("pD"), d("pS"), hd["node_child1"],
        hd["node_child2"], acc, S, active_mask=actd, merge_s_term=True, grad_log_pD=g_pD, grad_log_pS=g_pS, grad_mt=g_mt,
        accum_param_reductions=True, accum_mt_reduction=True, output_pibar_ud=True, output_pibar_side_active=True,
        pibar_side_threshold=0.0, mt_squeezed=t(mt), pibar_row_max=t(rmax), grad_mt_two_stage=True,
        skip_inactive_pibar_output_zero=True, item_idx=ints(item))
    torch.cuda.synchronize()
    want = np.zeros((C, S))
    np.add.at(want, SL, ref["direct_l"])
    np.add.at(want, SR, ref["direct_r"])
    close(acc, want, "direct adjoint rows")
    on = np.concatenate([ref["active_split"]] * 2)
    ond = torch.as_tensor(on).cuda()
    close(ud[ond], np.concatenate([ref["ud_l"], ref["ud_r"]])[on], "ud")
    close(A.reshape(-1)[ond], np.concatenate([ref["A_l"], ref["A_r"]])[on], "A")
    close(g_pD[0], ref["g_pD"].sum(0), "grad_log_pD")
    close(g_pS[0], ref["g_pS"].sum(0), "grad_log_pS")
    close(g_mt[0], (ref["g_mt_l"] + ref["g_mt_r"]).sum(0), "grad_mt")
    acc.zero_()
    gcol.zero_()
    wb.uniform_cross_pibar_vjp_tree_from_ud_fused(
        t(Pi), t(col), ud, A, ints(SL), ints(SR), acc, S, active_mask=actd, reduce_idx=ints(RED), pibar_row_max=t(rmax),
        skip_zero_sides=True, side_active=side, grad_col_log_probs=gcol, use_col_weights=weighted,
        side_active_threshold=0.0, **levels)
    torch.cuda.synchronize()
    want = np.zeros((C, S))
    np.add.at(want, SL, ref["tree_l"])
    np.add.at(want, SR, ref["tree_r"])
    close(acc, want, "Pibar VJP rows")
    close(gcol, ref["col_grad"], "grad_col")


@pytest.mark.parametrize("n", [15, 17, 1023, 1024, 1025, 2600])
@pytest.mark.parametrize("tdt", [torch.float32, torch.float64])
def test_column_sums_at_chunk_edges(n, tdt):
    """Row ranges of the wavefronts and chunks of the row sums: one launch up to 1024 rows, two above."""
    from kbench.core.kernels import _hip as H

    g = torch.Generator().manual_seed(n)
    S = 129
    xs = [torch.randn((n, S), generator=g, dtype=torch.float64).to(device="cuda", dtype=tdt) for _ in range(3)]
    base = torch.randn((S,), generator=g, dtype=torch.float64).to(device="cuda", dtype=tdt)
    want = [sum(x.double() for x in grp).sum(0) for grp in ((xs[0],), (xs[1], xs[2]), xs)]
    into, acc = base.clone(), [base.clone() for _ in want]
    H.sum_rows_into(into, xs[0])
    H.rows_sum_accum(list(zip(acc, ((xs[0],), (xs[1], xs[2]), tuple(xs)))))
    multi = H.rows_sum_multi([xs[0], (xs[1], xs[2])])
    torch.cuda.synchronize()
    print(f"[column sums] n={n} {tdt}", flush=True)
    # float64 sums of n values of size about 1 (n roundings of sqrt(n) 2^-53 each at the most), rounded once
    tol = 64 * n**1.5 * 2.0**-53 + (2.0**-24 * 6 * n**0.5 if tdt == torch.float32 else 0.0)
    assert torch.equal(into, acc[0])
    for got, ref in ((into, base.double() + want[0]), *zip(acc, (base.double() + w for w in want)), *zip(multi, want)):
        assert float((got.double() - ref).abs().max()) <= tol
