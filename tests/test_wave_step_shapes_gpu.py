"""``compute_wave_step`` at the edges of its launch shapes and of its two row forms, against the oracle.

A row whose span times its smallest constant (and weight) covers at most 120 binary orders
(float32; 1000 in float64) is swept in linear space, any other term by term in log space.  Rows of
both kinds, rows with -inf entries, a single finite entry or none, and two items whose constants
alternate over the rows share one launch.  That the switch lies where it must is the claim of
test_products_below_the_linear_range: in the other rows a transfer term hides what underflows.
"""

import numpy as np
import pytest
import torch

import kbench_oracle as O

pytestmark = pytest.mark.gpu

W = 6


def _case(leaves, dt, weighted, wide_consts, leaf):
    from kbench import synth

    rng = np.random.default_rng(leaves + 7 * weighted)
    tree = synth.yule_tree(leaves, rng)
    h = synth.state_helpers_from_tree(tree)
    S = tree.S
    rnd = lambda a: np.asarray(a).astype(dt).astype(np.float64)
    low = np.where(np.asarray(h["node_child1"]) < S, -8.0, 0.0)
    span = 90.0 if dt == np.float32 else 500.0
    Pi = -30.0 + rng.uniform(-12.0, 0.0, (W, S)) + low
    Pi[1, rng.random(S) < 0.5] = -np.inf
    Pi[2] = -20.0 + rng.uniform(-span, 0.0, S) + low
    Pi[2, 0] = -20.0
    Pi[3] = -np.inf
    Pi[4] = -np.inf
    Pi[4, S // 2] = -5.0
    dts = Pi - rng.uniform(1.0, 9.0, (W, S))
    dts[3] = -40.0 + low
    dts[5] = -np.inf
    c = {k: rng.uniform(-4.0, -0.5, (2, S)) for k in ("DL", "Ebar", "E", "SL1", "SL2", "leaf")}
    c["mt"] = rng.uniform(-12.0, -9.0, (2, S))
    if wide_consts:
        c["DL"][1, S // 3] = -span
    col = np.log2(rng.dirichlet(np.full(S, 50.0))) if weighted else np.full(S, -np.log2(S))
    c, Pi, dts, col = {k: rnd(v) for k, v in c.items()}, rnd(Pi), rnd(dts), rnd(col)
    items = np.arange(W) % 2
    leaf_state = rng.integers(0, S, W) if leaf else None
    consts = O.WaveConsts(mt=c["mt"], DL=c["DL"], Ebar=c["Ebar"], E=c["E"], SL1=c["SL1"], SL2=c["SL2"],
                          leaf_logp=c["leaf"], col=col, use_col_weights=weighted)
    return tree, h, S, Pi, dts, c, col, items, leaf_state, consts


def _device_sweep(case, dt, weighted, *, sweeps=1, store=True):
    from kbench.core.kernels import wave_step

    tree, h, S, Pi, dts, c, col, items, leaf_state, _ = case
    t = lambda a, d=dt: torch.as_tensor(np.ascontiguousarray(a), dtype=d, device="cuda")
    ints = lambda a: torch.as_tensor(np.asarray(a), dtype=torch.int64, device="cuda")
    bufs = [t(Pi), torch.full((W, S), 7.0, dtype=dt, device="cuda")]
    pibar, rmax = (torch.full(s, 7.0, dtype=dt, device="cuda") for s in ((W, S), (W,)))
    resid = torch.full((W,), 7.0, device="cuda") if sweeps == 1 else None
    consts = [t(c[k]) for k in ("mt", "DL", "Ebar", "E", "SL1", "SL2")]
    dev = dict(leaf_state_idx=ints(leaf_state if leaf_state is not None else np.zeros(W)), leaf_logp=t(c["leaf"]),
               item_idx=ints(items))
    topo = [ints(h[k]) for k in ("node_child1", "node_child2", "node_parent")]
    d = None if leaf_state is not None else t(dts)
    colt = t(col)
    for k in range(sweeps):
        wave_step.compute_wave_step(
            bufs[k % 2], bufs[(k + 1) % 2], pibar, 0, W, S, *consts, colt, *topo, int(h["max_ancestor_depth"]), d,
            **dev, pibar_row_max=rmax, store_final_pibar=store and k == sweeps - 1,
            has_leaf_term=leaf_state is not None, use_col_weights=weighted, pi_residual_out=resid)
    torch.cuda.synchronize()
    return bufs[sweeps % 2].cpu().numpy(), pibar.cpu().numpy(), rmax.cpu().numpy(), resid


# 4097 double rows need more LDS than the entry point allows (refused before any launch)
@pytest.mark.parametrize("leaves,kind", [(n, k) for n in (1, 2, 64, 65, 128, 129, 256, 257, 512, 513, 1024, 1025, 2049)
                                         for k in ("float32", "float64") if not (k == "float64" and n > 2048)])
def test_one_sweep_matches_oracle(leaves, kind):
    dt, tdt = (np.float32, torch.float32) if kind == "float32" else (np.float64, torch.float64)
    for weighted, wide_consts, leaf in ((False, False, False), (True, False, True), (False, True, True)):
        if leaves == 1 and weighted:
            continue  # one column: its weight is the whole distribution
        case = _case(leaves, dt, weighted, wide_consts, leaf)
        tree, h, S, Pi, dts, c, col, items, leaf_state, consts = case
        print(f"[sweep] S={S} {kind} weighted={weighted} wide_consts={wide_consts} leaf={leaf}", flush=True)
        out, pibar, rmax, resid = _device_sweep(case, tdt, weighted)
        otree = O.Tree.from_helpers(h)
        with np.errstate(all="ignore"):
            ref = O.wave_sweep(Pi, items, consts, otree, leaf_state=leaf_state, dts_r=None if leaf else dts)
            wcol = col if weighted else 0.0
            # each row's transfer term and its noise: a prefix-sum difference carries roundings of the
            # row's total (eps each, of which sqrt(S) survive), whatever the share of the others is
            eps = np.finfo(dt).eps
            noise = eps * (8.0 + 2.0 * np.sqrt(S))
            total = lambda x: np.exp2(x + wcol).sum(axis=1, keepdims=True)
            unit = np.exp2((c["E"] + c["mt"])[items]) * total(Pi)
            # a log2 value carries a few roundings of its own size and of its inputs'
            size = 4.0 * eps * np.nanmax(np.abs(np.where(np.isfinite(Pi), Pi, 0.0)), axis=1, keepdims=True) + 16.0 * eps
            y, y_ref = np.exp2(out.astype(np.float64)), np.exp2(ref)
            assert (np.abs(y - y_ref) <= size * y_ref + noise * unit).all(), "Pi"
            # Pibar and row_max belong to the rows written
            o64 = out.astype(np.float64)
            pb_ref, max_ref = O._pibar_from_pi(o64, col, c["mt"][items], otree, weighted)
            scale = np.exp2(c["mt"][items]) * total(o64)
            size = size + 4.0 * eps * np.abs(c["mt"][items])
            pb = np.exp2(pibar.astype(np.float64))
            assert (np.abs(pb - np.exp2(pb_ref)) <= size * np.exp2(pb_ref) + noise * scale).all(), "Pibar"
            assert np.allclose(rmax, max_ref, rtol=2.0 * eps, atol=0.0, equal_nan=True), "row_max"
            f = np.isfinite(out) & np.isfinite(Pi)
            want = np.abs(np.where(f, o64, 0.0) - np.where(f, Pi, 0.0)).max(axis=1)
        assert np.allclose(resid.cpu().numpy(), want, rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("leaves", [40, 400])
def test_float64_chain_is_bitwise_its_single_sweeps(leaves, monkeypatch):
    from kbench.core.kernels import wave_step

    case = _case(leaves, np.float64, True, False, False)
    one = _device_sweep(case, torch.float64, True, sweeps=3)
    monkeypatch.setattr(wave_step, "FUSE_SWEEPS", True)
    chain = _device_sweep(case, torch.float64, True, sweeps=3)
    for a, b in zip(one[:3], chain[:3]):
        assert np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("leaves,kind", [(n, k) for n in (1, 32, 64, 300, 512, 700, 1024, 1501)
                                         for k in ("float32", "float64")])
def test_nan_rows_stay_nan(leaves, kind):
    """A NaN entry reaches every entry that reads it, whatever else the row holds (the pattern of the oracle)."""
    dt, tdt = (np.float32, torch.float32) if kind == "float32" else (np.float64, torch.float64)
    for weighted, leaf, nan_dts in ((False, False, False), (False, False, True), (True, False, True),
                                    (False, True, False)):
        if leaves == 1 and weighted:
            continue
        tree, h, S, Pi, dts, c, col, items, leaf_state, consts = _case(leaves, dt, weighted, False, leaf)
        Pi[0] = np.nan
        Pi[1] = -np.inf
        Pi[1, S // 3] = np.nan
        Pi[2] = -20.0
        Pi[2, S - 1] = np.nan
        dts[1] = dts[3] = -np.inf
        if nan_dts:
            dts[0] = np.nan
            dts[3, S // 2] = np.nan
        if leaf:  # a NaN leaf value, a finite one in a NaN row, and one beside a NaN
            consts.leaf_logp[items[5], leaf_state[5]] = c["leaf"][items[5], leaf_state[5]] = np.nan
        case = (tree, h, S, Pi, dts, c, col, items, leaf_state, consts)
        print(f"[nan] S={S} {kind} weighted={weighted} leaf={leaf} nan_dts={nan_dts}", flush=True)
        out, pibar, _, resid = _device_sweep(case, tdt, weighted)
        with np.errstate(all="ignore"):
            ref = O.wave_sweep(Pi, items, consts, O.Tree.from_helpers(h), leaf_state=leaf_state,
                               dts_r=None if leaf else dts)
        assert np.isnan(ref[0]).all() and np.isnan(ref[1]).any() and not np.isnan(ref[4]).any()
        assert np.array_equal(np.isnan(out), np.isnan(ref)), "NaN"
        assert np.array_equal(np.isneginf(out), np.isneginf(ref)), "-inf"
        nan_row = np.isnan(ref).any(axis=1)
        assert np.isneginf(pibar[nan_row]).all(), "Pibar of a NaN row"
        # a NaN difference (of entries that are both above -inf) makes the residual NaN
        f = ~np.isneginf(ref) & ~np.isneginf(Pi)
        want = np.isnan(np.where(f, ref - np.where(f, Pi, 0.0), 0.0)).any(axis=1)
        assert np.array_equal(np.isnan(resid.cpu().numpy()), want), "residual"


@pytest.mark.parametrize("leaves,kind", [(n, k) for n in (2, 64, 65, 300, 600, 1024, 1501)
                                         for k in ("float32", "float64")])
def test_products_below_the_linear_range(leaves, kind):
    """Entries that only a product below the smallest normal number decides: compared in log2, where a
    flush to 0 shows as -inf.  Rows 0 and 1: one column of small weight and small Pi feeds the transfer
    term of all others, and the split term sets the row's largest entry (three factors, each of which
    alone would fit; two without weights).  Row 2: Pi over twice the format's range of exponents and no
    transfer.  Rows 3 and 4: small DL, Ebar, SL1 and SL2 times a small Pi.  Row 5: the products of row 0
    where the linear range just holds them."""
    dt, tdt = (np.float32, torch.float32) if kind == "float32" else (np.float64, torch.float64)
    f32 = dt == np.float32
    rng = np.random.default_rng(leaves)
    from kbench import synth

    tree = synth.yule_tree(leaves, rng)
    h = synth.state_helpers_from_tree(tree)
    S, root = tree.S, tree.root
    rnd = lambda a: np.asarray(a).astype(dt).astype(np.float64)
    col_low, em_low, pi_low = (-50.0, -50.0, -55.0) if f32 else (-390.0, -390.0, -390.0)
    for weighted in (False, True):
        c = {k: rng.uniform(-4.0, -0.5, (2, S)) for k in ("DL", "Ebar", "E", "SL1", "SL2", "leaf", "mt")}
        c["E"][:] = em_low
        Pi, dts = np.full((W, S), -np.inf), np.full((W, S), -np.inf)
        col = np.full(S, -np.log2(S))
        feed = 0  # a leaf: no column but itself has it among its ancestors
        if weighted:
            col[:] = -3.0
            col[feed] = col_low
        else:
            c["E"][:] = 2.0 * em_low
        c["mt"][:] = 0.0
        Pi[0, feed], dts[0, root] = -5.0 + pi_low, -5.0
        Pi[1, feed], dts[1, root] = -300.0 + pi_low, -300.0
        Pi[5, feed], dts[5, root] = -5.0, -5.0 - (3.0 if f32 else 200.0)
        # rows 2 to 4 are of items without transfers
        c["E"][0] = -np.inf
        items = np.array([1, 1, 0, 0, 0, 1])
        reach = 250.0 if f32 else 2100.0
        Pi[2] = -10.0 - np.linspace(0.0, reach, S)[rng.permutation(S)]
        Pi[3:5] = -20.0
        low = rng.permutation(S)[: max(1, S // 3)]
        Pi[3:5, low] = -20.0 - (70.0 if f32 else 600.0)
        for k, name in enumerate(("DL", "Ebar")):
            c[name][0, low] = -80.0 - k if f32 else -700.0 - k
        inner = np.nonzero(np.asarray(h["node_child1"]) < S)[0][: max(1, leaves // 3)]
        for name in ("SL1", "SL2"):
            c[name][0, inner] = -85.0 if f32 else -710.0
        c, Pi, dts, col = {k: rnd(v) for k, v in c.items()}, rnd(Pi), rnd(dts), rnd(col)
        consts = O.WaveConsts(mt=c["mt"], DL=c["DL"], Ebar=c["Ebar"], E=c["E"], SL1=c["SL1"], SL2=c["SL2"],
                              leaf_logp=c["leaf"], col=col, use_col_weights=weighted)
        case = (tree, h, S, Pi, dts, c, col, items, None, consts)
        print(f"[small] S={S} {kind} weighted={weighted}", flush=True)
        out, _, _, _ = _device_sweep(case, tdt, weighted)
        with np.errstate(all="ignore"):
            ref = O.wave_sweep(Pi, items, consts, O.Tree.from_helpers(h), dts_r=dts)
        if S > 3:
            assert np.isfinite(ref[:2]).sum() >= S  # (the test holds what it says it does)
        eps = np.finfo(dt).eps
        assert np.array_equal(np.isneginf(out), np.isneginf(ref)), (weighted, "entries of probability 0")
        f = np.isfinite(ref)
        # a log2 value carries a few roundings of its own size and of its inputs'
        tol = 4.0 * eps * (np.abs(ref[f]) + np.abs(Pi[np.isfinite(Pi)]).max()) + 16.0 * eps
        assert (np.abs(out[f] - ref[f]) <= tol).all(), (weighted, np.abs(out[f] - ref[f]).max())


def test_wide_rows_of_a_deep_tree():
    """Rows swept in log space on a tree of depth 1023: the oracle's values, at a few times the cost of rows
    swept in linear space (walking to the root from every entry took 50 times as long)."""
    from kbench import synth
    from kbench.core.kernels import wave_step

    L, rows = 1024, 600
    S = 2 * L - 1
    parent, c1, c2 = np.full(S, -1, np.int64), np.full(S, S, np.int64), np.full(S, S, np.int64)
    for j in range(L - 1):  # internal node L + j: leaf j + 1 and the internal node below (the lowest: two leaves)
        c1[L + j], c2[L + j] = (0, 1) if j == 0 else (j + 1, L + j - 1)
        parent[c1[L + j]] = parent[c2[L + j]] = L + j
    tree = synth._finish_tree(synth.SpeciesTree(L, parent, c1, c2, np.zeros(S)))
    h = synth.state_helpers_from_tree(tree)
    assert h["max_ancestor_depth"] == L
    rng = np.random.default_rng(5)
    f32 = lambda a: np.asarray(a, np.float32).astype(np.float64)
    c = {k: f32(rng.uniform(-4.0, -0.5, (1, S))) for k in ("DL", "Ebar", "E", "SL1", "SL2", "leaf", "mt")}
    col = f32(np.full(S, -np.log2(S)))
    consts = O.WaveConsts(mt=c["mt"], DL=c["DL"], Ebar=c["Ebar"], E=c["E"], SL1=c["SL1"], SL2=c["SL2"],
                          leaf_logp=c["leaf"], col=col, use_col_weights=False)
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float32, device="cuda")
    ints = lambda a: torch.as_tensor(np.asarray(a), dtype=torch.int64, device="cuda")
    dev = [t(c[k]) for k in ("mt", "DL", "Ebar", "E", "SL1", "SL2")]
    topo = [ints(h[k]) for k in ("node_child1", "node_child2", "node_parent")]
    rest = dict(leaf_state_idx=ints(np.zeros(rows)), leaf_logp=t(c["leaf"]), item_idx=ints(np.zeros(rows)),
                pibar_row_max=t(np.zeros(rows)), store_final_pibar=False, has_leaf_term=False, use_col_weights=False)
    took = {}
    for span in (30.0, 200.0):
        Pi = f32(-10.0 - rng.uniform(0.0, span, (rows, S)))
        src, out, colt = t(Pi), t(np.zeros((rows, S))), t(col)
        sweep = lambda: wave_step.compute_wave_step(src, out, out, 0, rows, S, *dev, colt, *topo, L, None, **rest)
        sweep()
        times = []
        for _ in range(7):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            sweep()
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        took[span] = float(np.median(times))
        with np.errstate(all="ignore"):
            ref = O.wave_sweep(Pi, np.zeros(rows, np.int64), consts, O.Tree.from_helpers(h))
        eps = np.finfo(np.float32).eps
        unit = np.exp2((c["E"] + c["mt"])[0]) * np.exp2(Pi).sum(axis=1, keepdims=True)  # the transfer term's noise
        y, y_ref = np.exp2(out.cpu().numpy().astype(np.float64)), np.exp2(ref)
        size = 4.0 * eps * np.abs(Pi).max() + 16.0 * eps
        assert (np.abs(y - y_ref) <= size * y_ref + eps * (8.0 + 2.0 * np.sqrt(S)) * unit).all(), span
    print(f"[deep tree] {took}", flush=True)
    assert took[200.0] <= 8.0 * took[30.0]


@pytest.mark.parametrize("leaves,kind,rows", [
    (64, "float32", 14000), (300, "float32", 4000), (512, "float32", 2600), (1024, "float32", 2000),
    (1501, "float32", 1100), (2049, "float32", 700), (64, "float64", 14000), (300, "float64", 4000),
    (512, "float64", 2600), (1024, "float64", 1500), (1501, "float64", 800)])
def test_rows_do_not_depend_on_their_predecessors(leaves, kind, rows):
    """More rows than workgroups: each walks rows of several items, with and without room for the linear
    form, and of none but -inf.  The same rows in another order give the same bits; a sample is the oracle's."""
    from kbench import synth
    from kbench.core.kernels import wave_step

    dt, tdt = (np.float32, torch.float32) if kind == "float32" else (np.float64, torch.float64)
    rng = np.random.default_rng(leaves)
    tree = synth.yule_tree(leaves, rng)
    h = synth.state_helpers_from_tree(tree)
    S, G = tree.S, 5
    print(f"[predecessors] S={S} {kind} rows={rows}", flush=True)
    rnd = lambda a: np.asarray(a).astype(dt).astype(np.float64)
    c = {k: rnd(rng.uniform(-6.0, -0.5, (G, S))) for k in ("DL", "Ebar", "E", "SL1", "SL2", "leaf", "mt")}
    c["DL"][4] = rnd(c["DL"][4] - (150.0 if dt == np.float32 else 1100.0))  # no row of this item is linear
    c["Ebar"][4] = -np.inf
    col = rnd(np.log2(rng.dirichlet(np.full(S, 50.0))))
    g = torch.Generator(device="cuda").manual_seed(leaves)
    Pi = -10.0 - 30.0 * torch.rand((rows, S), generator=g, device="cuda", dtype=tdt)
    kinds = torch.randint(0, 6, (rows,), generator=g, device="cuda")
    Pi[kinds == 4] *= 6.0 if dt == np.float32 else 50.0
    Pi[kinds == 5] = -float("inf")
    dts = Pi - 3.0
    items = torch.randint(0, G, (rows,), generator=g, device="cuda")
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=tdt, device="cuda")
    ints = lambda a: torch.as_tensor(np.asarray(a), dtype=torch.int64, device="cuda")
    dev, colt, leaf = [t(c[k]) for k in ("mt", "DL", "Ebar", "E", "SL1", "SL2")], t(col), t(c["leaf"])
    topo, zero = [ints(h[k]) for k in ("node_child1", "node_child2", "node_parent")], ints(np.zeros(rows))

    def sweep(order):
        out, pibar = torch.empty_like(Pi), torch.empty_like(Pi)
        rmax = torch.empty((rows,), dtype=tdt, device="cuda")
        wave_step.compute_wave_step(
            Pi[order].contiguous(), out, pibar, 0, rows, S, *dev, colt, *topo, int(h["max_ancestor_depth"]),
            dts[order].contiguous(), leaf_state_idx=zero, leaf_logp=leaf, item_idx=items[order].contiguous(),
            pibar_row_max=rmax, store_final_pibar=True, has_leaf_term=False, use_col_weights=True)
        back = torch.argsort(order)
        return out[back], pibar[back], rmax[back]

    a = sweep(torch.arange(rows, device="cuda"))
    b = sweep(torch.randperm(rows, generator=g, device="cuda"))
    for x, y in zip(a, b):
        assert torch.equal(x, y)
    pick = rng.choice(rows, 40, replace=False)
    take = lambda x: x[torch.as_tensor(pick, device="cuda")].double().cpu().numpy()
    consts = O.WaveConsts(mt=c["mt"], DL=c["DL"], Ebar=c["Ebar"], E=c["E"], SL1=c["SL1"], SL2=c["SL2"],
                          leaf_logp=c["leaf"], col=col, use_col_weights=True)
    P, it = take(Pi), items.cpu().numpy()[pick]
    with np.errstate(all="ignore"):
        ref = O.wave_sweep(P, it, consts, O.Tree.from_helpers(h), dts_r=take(dts))
        unit = np.exp2((c["E"] + c["mt"])[it]) * np.exp2(P + col).sum(axis=1, keepdims=True)  # the transfer's noise
    eps = np.finfo(dt).eps
    y, y_ref = np.exp2(take(a[0])), np.exp2(ref)
    size = 4.0 * eps * np.abs(P[np.isfinite(P)]).max() + 16.0 * eps
    assert (np.abs(y - y_ref) <= size * y_ref + eps * (8.0 + 2.0 * np.sqrt(S)) * unit).all()
