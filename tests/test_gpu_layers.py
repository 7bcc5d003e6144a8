"""End-to-end parity of the drop-in layers on the GPU: CompressgnnData -> CompressGraph ->
KPropagate forward/backward against (a) the CPU oracle's 4-stage chain on the same blocks
and (b) the plain, uncompressed A^T x of the same graph; Compressgnn_Cluster /
Compressgnn_Reconstruct forward/backward against the oracle and torch autograd of the
index_select composition (the checks of the reference's tests/test_transformation.py)."""
import gc
import os
import sys

import numpy as np
import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path[:0] = [os.path.join(ROOT, "compressgnn_amd"), os.path.join(ROOT, "compressgnn_amd", "layer"),
                os.path.join(ROOT, "compressgnn_amd", "loader")]

import oracle
from util import assert_no_less_accurate, assert_within

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _np_blocks(graph):
    def csr(g):
        rp, ci, val = g.csr()
        return rp.cpu().numpy(), ci.cpu().numpy(), val.cpu().numpy()

    def csc(g):
        cp, row, val = g.csc()
        return cp.cpu().numpy(), row.cpu().numpy(), val.cpu().numpy()

    fwd = dict(v2v=csr(graph.v2v_graph), v2r=csr(graph.v2r_graph), r2v=csr(graph.r2v_graph),
               r2r=[csr(g) for g in graph.r2r_graph])
    bwd = dict(v2v_t=csc(graph.v2v_graph), v2r_t=csc(graph.v2r_graph), r2v_t=csc(graph.r2v_graph),
               r2r_t=[csc(g) for g in graph.r2r_graph])
    return fwd, bwd


def _make_data(kind, F, normalize=True, freq=16, seed=0):
    import compressgnn_offline as off
    from CompressgnnData import CompressgnnData
    rng = np.random.default_rng(seed)
    if kind == "chung_lu":
        v, e = off.gen_chung_lu(2708, 10500, 2.5, seed)
    elif kind == "copy":
        v, e = off.gen_copy_model(6000, 9.8, 0.7, seed)
    elif kind == "blocks":
        n = 64
        v = np.arange(n + 1, dtype=np.int64) * 32
        e = np.tile(np.arange(32, dtype=np.int64), n)
    V = len(v) - 1
    x = rng.standard_normal((V, F)).astype(np.float32)
    mask = np.ones(V, dtype=bool)
    data = CompressgnnData(x, (v, e), np.zeros(V, np.int64), mask, mask, mask, add_self_loop=True,
                           normalize=normalize, graph_type="csr", min_pair_frequency=freq)
    return data, (v, e)


def _plain_transpose_product(v, e, x, normalize):
    """out = A_hat^T x of the uncompressed graph with self loops and (optionally)
    symmetric normalisation, in float64."""
    import compressgnn_offline as off
    v2, e2 = off.add_self_loop_csr(v, e)
    V = len(v2) - 1
    src = np.repeat(np.arange(V), np.diff(v2))
    if normalize:
        d = off.get_norm_degree(e2, V).astype(np.float64)
        w = d[src] * d[e2]
    else:
        w = np.ones(len(e2))
    out = np.zeros((V, x.shape[1]))
    np.add.at(out, e2, w[:, None] * x[src].astype(np.float64))
    return out


def _plain_product(v, e, g, normalize):
    """gx = A_hat g of the same graph (the gradient of _plain_transpose_product), in float64."""
    import compressgnn_offline as off
    v2, e2 = off.add_self_loop_csr(v, e)
    V = len(v2) - 1
    src = np.repeat(np.arange(V), np.diff(v2))
    if normalize:
        d = off.get_norm_degree(e2, V).astype(np.float64)
        w = d[src] * d[e2]
    else:
        w = np.ones(len(e2))
    out = np.zeros((V, g.shape[1]))
    np.add.at(out, src, w[:, None] * g[e2].astype(np.float64))
    return out


@pytest.mark.parametrize("kind,freq", [("chung_lu", 16), ("chung_lu", 3), ("copy", 3), ("blocks", 16)])
@pytest.mark.parametrize("normalize", [True, False])
@pytest.mark.parametrize("F", [128, 16])
def test_propagate_forward_backward(kind, freq, normalize, F):
    from KPropagate import KPropagate
    data, (v, e) = _make_data(kind, F, normalize, freq)
    graph = data.edge_index
    fwd_blocks, bwd_blocks = _np_blocks(graph)
    x_np = data.x.numpy().copy()
    if kind != "chung_lu" or freq == 3:
        assert data.rule_cnt > 0
    want = oracle.compress_spmm_forward(fwd_blocks, x_np) if data.rule_cnt else oracle.spmm(*fwd_blocks["v2v"], x_np)
    plain = _plain_transpose_product(v, e, x_np, normalize)
    # the oracle's compressed chain equals the uncompressed product (re-association only)
    np.testing.assert_allclose(want, plain, rtol=2e-4, atol=2e-5 if normalize else 2e-3)

    data.to(DEV)
    prop = KPropagate()
    x = data.x.detach().clone().requires_grad_()
    out = prop(x, data.edge_index, None, data.vertex_cnt, data.rule_cnt)
    g_np = np.random.default_rng(5).standard_normal(out.shape).astype(np.float32)
    (gx,) = torch.autograd.grad(out, x, torch.from_numpy(g_np).to(DEV))
    torch.cuda.synchronize()
    want_gx = (oracle.compress_spmm_backward(bwd_blocks, g_np) if data.rule_cnt
               else oracle.spmm(*bwd_blocks["v2v_t"], g_np))
    if normalize:
        assert_within(out.detach().cpu().numpy(), want, rtol=1e-5, atol=1e-6)
        assert_within(gx.cpu().numpy(), want_gx, rtol=1e-5, atol=1e-6)
    else:
        # unit weights: sums of up to hundreds of O(1) terms, where two summation orders differ
        # by more than 1e-6 absolute.  The bar that can fail: the kernels are no further from
        # the float64 product than the oracle's sequential fp32 chain is.
        plain_g = _plain_product(v, e, g_np, normalize)
        assert_no_less_accurate(out.detach().cpu().numpy(), want, plain)
        assert_no_less_accurate(gx.cpu().numpy(), want_gx, plain_g)
        assert_within(out.detach().cpu().numpy(), want, rtol=1e-5, atol=1e-4)
        assert_within(gx.cpu().numpy(), want_gx, rtol=1e-5, atol=1e-4)
    # adjoint identity <A x, g> == <x, A^T g> in float64 on the GPU results
    lhs = float((out.detach().cpu().numpy().astype(np.float64) * g_np).sum())
    rhs = float((x_np.astype(np.float64) * gx.cpu().numpy()).sum())
    assert abs(lhs - rhs) <= 1e-4 * max(1.0, abs(lhs))


@pytest.mark.parametrize("kind,freq", [("chung_lu", 3), ("copy", 3), ("chung_lu", 16)])
@pytest.mark.parametrize("normalize", [True, False])
def test_coo_multi_phase_propagate(kind, freq, normalize):
    """graph_type="coo": KPropagate over the per-phase edge lists, forward and gradient,
    against the oracle's sequential scatter-add over the same phases (the reference's
    gather + scatter loop), the CompressGraph path on the same graph, and the adjoint
    identity.  Tolerance 1e-5 relative / 1e-6 absolute on normalised weights."""
    import compressgnn_offline as off
    import prep_oracle
    from CompressgnnData import CompressgnnData
    from KPropagate import KPropagate
    F = 64
    csr_data, (v, e) = _make_data(kind, F, normalize, freq)
    V = len(v) - 1
    src, dst = off.csr2coo(v, e)
    m = np.ones(V, bool)
    data = CompressgnnData(csr_data.x.numpy(), (src, dst), np.zeros(V, np.int64), m, m, m, add_self_loop=True,
                           normalize=normalize, graph_type="coo", min_pair_frequency=freq)
    assert (data.vertex_cnt, data.rule_cnt) == (csr_data.vertex_cnt, csr_data.rule_cnt)
    x_np = data.x.numpy().copy()
    phases = [t.numpy() for t in data.edge_index]
    weights = [t.numpy() for t in data.edge_weight]
    want = prep_oracle.coo_propagate(x_np, phases, weights, data.vertex_cnt, data.rule_cnt)
    g_np = np.random.default_rng(9).standard_normal(want.shape).astype(np.float32)
    # gradient oracle: the transposed phases in reverse order
    full = np.concatenate([g_np, np.zeros((data.rule_cnt, F), np.float32)])
    for edges, w in reversed(list(zip(phases[1:], weights[1:]))):
        np.add.at(full, edges[0], w.reshape(-1, 1) * full[edges[1]])
    want_gx = np.zeros_like(x_np)
    np.add.at(want_gx, phases[0][0], weights[0].reshape(-1, 1) * full[phases[0][1]])

    data.to(DEV)
    csr_data.to(DEV)
    prop = KPropagate()
    x = data.x.detach().clone().requires_grad_()
    out = prop(x, data.edge_index, data.edge_weight, data.vertex_cnt, data.rule_cnt)
    assert out.shape == (V, F)
    (gx,) = torch.autograd.grad(out, x, torch.from_numpy(g_np).to(DEV))
    again = prop(x, data.edge_index, data.edge_weight, data.vertex_cnt, data.rule_cnt)  # cached plan
    torch.cuda.synchronize()
    tol = dict(rtol=1e-5, atol=1e-6) if normalize else dict(rtol=1e-5, atol=1e-4)
    assert_within(out.detach().cpu().numpy(), want, **tol)
    assert_within(gx.cpu().numpy(), want_gx, **tol)
    if not normalize:  # the widened bound alone proves little: also no further from float64 than the oracle
        assert_no_less_accurate(out.detach().cpu().numpy(), want, _plain_transpose_product(v, e, x_np, normalize))
        assert_no_less_accurate(gx.cpu().numpy(), want_gx, _plain_product(v, e, g_np, normalize))
    assert torch.equal(out, again)
    via_graph = KPropagate()(csr_data.x, csr_data.edge_index, None, csr_data.vertex_cnt, csr_data.rule_cnt)
    assert_within(out.detach().cpu().numpy(), via_graph.cpu().numpy(), **tol)
    lhs = float((out.detach().cpu().numpy().astype(np.float64) * g_np).sum())
    rhs = float((x_np.astype(np.float64) * gx.cpu().numpy()).sum())
    assert abs(lhs - rhs) <= 1e-4 * max(1.0, abs(lhs))
    with pytest.raises(ValueError):
        prop(x, data.edge_index, data.edge_weight)  # vertex_cnt / rule_cnt are required


@pytest.mark.parametrize("fuse", [True, False])
@pytest.mark.parametrize("method", ["row_schedule", "nnz_schedule", "auto", "rowbalance_rowcache"])
def test_propagate_schedules_agree(fuse, method):
    from CompressgnnSPMM import compress_spmm
    data, _ = _make_data("copy", 64, True, 3)
    fwd_blocks, _ = _np_blocks(data.edge_index)
    want = oracle.compress_spmm_forward(fwd_blocks, data.x.numpy())
    data.to(DEV)
    data.edge_index.fold_levels = method != "row_schedule"  # one launch per level: the oracle's order of sums
    data.edge_index.keep_split_blocks = not fuse
    plan = data.edge_index.plan()
    assert all(b.offloaded for b in data.edge_index.blocks())  # the device holds the plan's arrays only
    plan.fuse_final, plan.method = fuse, method
    out = compress_spmm(data.edge_index, data.x)
    torch.cuda.synchronize()
    assert_within(out.cpu().numpy(), want)
    if method == "row_schedule":
        assert np.array_equal(out.cpu().numpy(), want)  # sequential sums in every stage


@pytest.mark.parametrize("F", [16, 64, 256, 512])
@pytest.mark.parametrize("method,fold,fuse", [("auto", True, True), ("nnz_schedule", True, True),
                                              ("nnz_schedule", False, False), ("row_schedule", False, True),
                                              ("row_schedule", False, False)])
def test_plan_feature_sweep(F, method, fold, fuse):
    """The widths of the feature sweep through the propagation plan itself, forward and
    gradient: folded rule stage and fused two-source vertex stages (F = 512 takes two feature
    tiles per lane), both schedules, and the launch-per-level / two-launch forms, against the
    oracle's 4-stage chain at 1e-5 relative / 1e-6 absolute.  A forced row schedule with one
    launch per level sums in the oracle's order: same bits."""
    data, _ = _make_data("copy", F, True, 3, seed=F)
    graph = data.edge_index
    assert data.rule_cnt > 0 and graph.step >= 1
    fwd_blocks, bwd_blocks = _np_blocks(graph)
    x_np = data.x.numpy().copy()
    g_np = np.random.default_rng(F).standard_normal(x_np.shape).astype(np.float32)
    want = oracle.compress_spmm_forward(fwd_blocks, x_np)
    want_g = oracle.compress_spmm_backward(bwd_blocks, g_np)
    data.to(DEV)
    graph.fold_levels, graph.keep_split_blocks = fold, not fuse
    plan = graph.plan()
    assert graph.levels_folded == fold
    plan.fuse_final, plan.method = fuse, method
    out = plan.forward(data.x)
    gx = plan.backward(torch.from_numpy(g_np).to(DEV))
    torch.cuda.synchronize()
    assert_within(out.cpu().numpy(), want, rtol=1e-5, atol=1e-6)
    assert_within(gx.cpu().numpy(), want_g, rtol=1e-5, atol=1e-6)
    if method == "row_schedule":
        assert np.array_equal(out.cpu().numpy(), want) and np.array_equal(gx.cpu().numpy(), want_g)
    if not fuse:
        with pytest.raises(RuntimeError):  # a plan built without the split blocks says so
            other, _ = _make_data("copy", 16, True, 3, seed=F)
            other.to(DEV)
            other.edge_index.plan().fuse_final = False

@pytest.mark.parametrize("F,one_launch", [(8, (True, True)), (128, (True, True)), (384, (False, True)), (1024, (False, False))])
def test_rules_multiplied_out_or_in_stages(F, one_launch):
    """A web graph of 60,000 vertices on both sides of the line from which a propagation runs its rule stage: AUTO against
    the stages themselves (a forced schedule runs them), forward and gradient, and the propagation from representatives
    gives the bits of the plain one on either side."""
    import compressgnn_offline as off
    from CompressgnnData import CompressgnnData
    v, e = off.gen_copy_model(60000, 9.8, 0.7, 3)
    V, mask = len(v) - 1, np.ones(len(v) - 1, bool)
    data = CompressgnnData(np.zeros((V, 1), np.float32), (v, e), np.zeros(V, np.int64), mask, mask, mask, graph_type="csr")
    data.to(DEV)
    plan = data.edge_index.plan()
    gen = torch.Generator(device=DEV).manual_seed(F)
    x, g = (torch.randn(V, F, device=DEV, generator=gen) for _ in range(2))
    plan.timed_stages = ["*"]
    out, grad = plan.forward(x), plan.backward(g)
    torch.cuda.synchronize()
    names = [name for name, _ in plan.take_stage_times()]
    assert names == [n for way, alone in zip(("fwd", "bwd"), one_launch) for n in ([] if alone else [way + ".rules"]) + [way + ".final"]]
    plan.timed_stages = []
    index = torch.randint(0, 900, (V,), device=DEV, generator=gen)
    reps = torch.randn(900, F, device=DEV, generator=gen)
    assert torch.equal(plan.forward_gathered(reps, index), plan.forward(reps.index_select(0, index)))
    plan.method = "nnz_schedule"
    # the same products in another order, and one more rounding of a weight: 2^-24 of the sum of absolute values per step
    assert_within(out.cpu().numpy(), plan.forward(x).cpu().numpy(), rtol=1e-5, atol=1e-6)
    assert_within(grad.cpu().numpy(), plan.backward(g).cpu().numpy(), rtol=1e-5, atol=1e-6)


def _plan_over(dtype, near, far, rules):
    """A propagation plan over device arrays of its own, [near | far] its vertex stage and `rules` its rule stage (scipy
    matrices): (plan, the values of the rule stage, of its transpose, of the vertex stage, of its transpose)."""
    import scipy.sparse as sp
    import compressgnn_runtime as rt
    (R, V), values, blocks = rules.shape, [], []
    for m in (rules, far.T, sp.hstack([near, far]), sp.hstack([near.T, rules.T])):
        m = m.tocsr()
        m.sort_indices()
        rowptr, col, val = (torch.from_numpy(a.astype(kind)).to(DEV)
                            for a, kind in ((m.indptr, np.int32), (m.indices, np.int32), (m.data, dtype)))
        values.append(val)
        blocks.append(rt.DeviceCsr(rowptr, col, val, m.shape[0], m.shape[1], torch.device(DEV), 32))
    plan = rt.PropagationPlan(V, R, blocks[0], [], blocks[1], [])
    plan.set_vertex_stages(blocks[2], blocks[3])
    return plan, values


def _random_stages(seed, near_is=None, far_is=None, rules_is=None, V=300, R=24):
    import scipy.sparse as sp
    rng = np.random.default_rng(seed)
    made = []
    for shape, density, value in (((V, V), 0.02, near_is), ((V, R), 0.1, far_is), ((R, V), 0.05, rules_is)):
        m = sp.random(*shape, density, "csr", random_state=rng, dtype=np.float64)
        if value is not None:
            m.data[:] = value
        made.append(m)
    return made


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("factors", ["small", "large", "infinite", "far_apart", "ordinary"])
def test_weights_whose_products_leave_the_range(dtype, factors):
    """Values of two stages whose products have no place in the type, though the sums of the stages have: such a plan runs
    its stages, others a launch alone, forward and gradient."""
    tiny, huge = (1e-25, 1e25) if dtype == np.float32 else (1e-180, 1e180)
    w, v, scale = dict(small=(tiny, tiny, huge), large=(huge, huge, tiny), infinite=(np.inf, tiny, huge),
                       far_apart=(tiny, huge, 1.0), ordinary=(0.3, 0.7, 1.0))[factors]
    in_range = factors in ("far_apart", "ordinary")
    near, far, rules = _random_stages(5, None if in_range else 0.0, w, v)
    plan, _ = _plan_over(dtype, near, far, rules)
    plan.timed_stages = ["*"]
    x_np = ((0.5 + np.random.default_rng(3).random((300, 12))) * scale).astype(dtype)
    x = torch.from_numpy(x_np).to(DEV)
    chains = ((near, far, rules), (near.T, rules.T, far.T))
    for got, (vertices, second, first) in zip((plan.forward(x), plan.backward(x)), chains):
        got = got.cpu().numpy()
        if in_range:  # sums of up to 40 positive terms, three roundings each
            want = vertices @ x_np.astype(np.float64) + second @ (first @ x_np.astype(np.float64))
            np.testing.assert_allclose(got, want, rtol=64 * np.finfo(dtype).eps)
            continue
        ones = lambda m: (m != 0).astype(np.float64)
        paths = (ones(second) @ (ones(first) @ np.ones(300)))[:, None]
        if factors == "infinite":
            assert np.isinf(got[paths[:, 0] > 0]).all()
            continue
        # every term is w * v * x with x in [0.5, 1.5] scale
        size = float(w) * (float(v) * scale)
        assert (got >= 0.49 * size * paths).all() and (got <= 1.51 * size * paths).all() and paths.any()
    names = [name for name, _ in plan.take_stage_times()]
    assert names == (["fwd.final", "bwd.final"] if in_range else ["fwd.rules", "fwd.final", "bwd.rules", "bwd.final"])


@pytest.mark.parametrize("which", [0, 1, 2, 3])
def test_values_written_after_the_plan_was_made(which):
    """The values of a plan's blocks may be the caller's own tensors.  A product behind a write to one of them uses what
    stands there then, also where the products before it ran as one launch."""
    near, far, rules = _random_stages(6)
    plan, values = _plan_over(np.float32, near, far, rules)
    x_np = np.random.default_rng(4).standard_normal((300, 12)).astype(np.float32)
    x = torch.from_numpy(x_np).to(DEV)
    plan.forward(x), plan.backward(x)
    values[which].mul_(3.0)
    by = [3.0 if k == which else 1.0 for k in range(4)]
    want = by[2] * (near @ x_np + far @ (by[0] * (rules @ x_np)))
    want_g = by[3] * (near.T @ x_np + rules.T @ (by[1] * (far.T @ x_np)))
    for _ in range(2):
        assert_within(plan.forward(x).cpu().numpy(), want, rtol=1e-5, atol=2e-5)
        assert_within(plan.backward(x).cpu().numpy(), want_g, rtol=1e-5, atol=2e-5)


def test_columns_written_between_the_replays_of_a_recorded_making():
    """A graph whose capture holds a plan's first product of the multiplied-out form makes the block with every replay.  Where
    the columns have changed meanwhile, so that it comes to more or fewer entries than there is room for, it stays inside its
    arrays; and with the columns as they were its replays are right again."""
    near, far, rules = _random_stages(8)
    plan, _ = _plan_over(np.float32, near, far, rules)
    x = torch.randn(300, 12, device=DEV)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        recorded = plan.forward(x), plan.backward(x)
    want = plan.forward(x), plan.backward(x)
    columns = plan.vertex_stage.colidx
    kept = columns.clone()
    for fewer in (None, True, False):
        if fewer is not None:  # vertices alone; rules alone
            columns.copy_(torch.randint(0, 300, kept.shape, device=DEV) if fewer else torch.randint(300, 324, kept.shape, device=DEV))
            graph.replay()
            torch.cuda.synchronize()
            assert recorded[0].shape == want[0].shape
        columns.copy_(kept)
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(recorded, want))


def test_plans_over_values_of_other_types():
    """Values of a type that no product takes are refused by the product, as ever, and not while the plan is made."""
    plan, _ = _plan_over(np.float16, *_random_stages(7))
    x = torch.randn(300, 12, device=DEV)
    for mat in (x, x.half()):
        with pytest.raises(RuntimeError):
            plan.forward(mat)


def _requested():
    return torch.cuda.memory_stats()["requested_bytes.all.current"]


def _web_graph_plan(vertices):
    import compressgnn_offline as off
    from CompressgnnData import CompressgnnData
    v, e = off.gen_copy_model(vertices, 9.8, 0.7, 3)
    V, mask = len(v) - 1, np.ones(len(v) - 1, bool)
    data = CompressgnnData(np.zeros((V, 1), np.float32), (v, e), np.zeros(V, np.int64), mask, mask, mask, graph_type="csr")
    return data.to(DEV).edge_index.plan()


def test_multiplied_out_blocks_are_made_for_the_products_that_take_them():
    """A plan holds its stages alone until a product takes the multiplied-out form, whose columns and values are 8 bytes an
    entry."""
    plan = _web_graph_plan(60000)
    wide, narrow = torch.randn(plan.vertex_stage.rows, 1024, device=DEV), torch.randn(plan.vertex_stage.rows, 8, device=DEV)
    entries = plan.vertex_stage.nnz + plan.vertex_stage_t.nnz
    plan.forward(wide), plan.backward(wide)  # with the tables of the stages
    before = _requested()
    first = plan.forward(narrow), plan.backward(narrow)
    assert _requested() - before >= 8 * entries
    assert all(torch.equal(a, b) for a, b in zip(first, (plan.forward(narrow), plan.backward(narrow))))
    other = torch.cuda.Stream()  # the blocks are finished: a stream that waits for nothing may use them
    with torch.cuda.stream(other):
        got = plan.forward(narrow)
    torch.cuda.synchronize()
    assert torch.equal(got, first[0])


@pytest.mark.parametrize("F", [1024, 8])
def test_representatives_compose_the_blocks_that_their_width_takes(F):
    """A new index sends the columns of the stages or of the multiplied-out block through it, 4 bytes an entry, and not of
    both; a product of the other width over the same index, also one that is recorded, has the bits of the plain one."""
    plan = _web_graph_plan(60000)
    V = plan.vertex_stage.rows
    index = torch.randint(0, 900, (V,), device=DEV)
    reps, other = torch.randn(900, F, device=DEV), torch.randn(900, 1032 - F, device=DEV)
    want, want_other = (plan.forward(r.index_select(0, index)) for r in (reps, other))
    torch.cuda.synchronize()
    before = _requested()
    got = plan.forward_gathered(reps, index)
    held = _requested() - before - 4 * got.numel()
    assert torch.equal(got, want)
    # the multiplied-out block has 1.05 entries for one of the stages
    assert held < 1.3 * 4 * (plan.r2v.nnz + plan.vertex_stage.nnz)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        recorded = plan.forward_gathered(other, index)
    for _ in range(3):
        assert torch.equal(plan.forward_gathered(other, index), want_other)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(recorded, want_other)
    with pytest.raises(RuntimeError, match="outside"):
        plan.forward_gathered(reps, torch.full((V,), 900, device=DEV))


def test_rule_levels_are_stored_without_their_padding():
    """One launch per level (the form kept for hierarchies too deep to fold): the reference pads
    every level to all R rule rows (src/offline/csrc/partition.h:175-203); the device form of a level
    holds only the rules of that level, each with the row it updates, and the chain over the
    levels gives the oracle's bits in a forced row schedule, forward and gradient."""
    import compressgnn_offline as off
    from CompressgnnData import CompressgnnData
    v, e = off.gen_copy_model(3000, 9.8, 0.7, 2)
    V = len(v) - 1
    m = np.ones(V, bool)
    rng = np.random.default_rng(8)
    x_np = rng.standard_normal((V, 48)).astype(np.float32)
    data = CompressgnnData(x_np, (v, e), np.zeros(V, np.int64), m, m, m, graph_type="csr", min_pair_frequency=3,
                           threshold=0, max_depth=8, min_edge=0, verbose=False)
    graph = data.edge_index
    assert graph.step >= 2, "the fixture should have several rule levels"
    fwd_blocks, bwd_blocks = _np_blocks(graph)
    g_np = rng.standard_normal(x_np.shape).astype(np.float32)
    want, want_g = oracle.compress_spmm_forward(fwd_blocks, x_np), oracle.compress_spmm_backward(bwd_blocks, g_np)
    per_level = [int(np.count_nonzero(np.diff(b[0]))) for b in fwd_blocks["r2r"]]
    data.to(DEV)
    graph.fold_levels = False
    plan = graph.plan()
    assert not graph.levels_folded and len(plan.r2r) == graph.step == len(plan.r2r_t)
    R = data.rule_cnt
    assert [b.rows for b in plan.r2r] == per_level and all(b.out_rows == R and b.rows < R for b in plan.r2r + plan.r2r_t)
    plan.method = "row_schedule"
    out, gx = plan.forward(data.x), plan.backward(torch.from_numpy(g_np).to(DEV))
    assert np.array_equal(out.cpu().numpy(), want) and np.array_equal(gx.cpu().numpy(), want_g)
    plan.method = "nnz_schedule"
    assert_within(plan.forward(data.x).cpu().numpy(), want, rtol=1e-5, atol=1e-6)
    assert_within(plan.backward(torch.from_numpy(g_np).to(DEV)).cpu().numpy(), want_g, rtol=1e-5, atol=1e-6)


def test_propagation_replays_from_a_captured_graph():
    """Forward and gradient propagation make no host read, no memset and no allocation outside
    torch's allocator, so a step can be captured in a graph; every replay, with eager work and
    synchronisations in between and new values in the captured inputs, gives the bits of the eager step."""
    data, _ = _make_data("copy", 64, True, 3, seed=4)
    data.to(DEV)
    plan = data.edge_index.plan()
    V = data.vertex_cnt
    gen = torch.Generator(device=DEV)
    gen.manual_seed(9)
    x = torch.randn(V, 64, device=DEV, generator=gen)
    g = torch.randn(V, 64, device=DEV, generator=gen)

    def step():
        return plan.forward(x), plan.backward(g)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out_graph, gx_graph = step()
    for _ in range(3):
        x.copy_(torch.randn(V, 64, device=DEV, generator=gen))
        g.copy_(torch.randn(V, 64, device=DEV, generator=gen))
        assert torch.isfinite((x * 2).sum()).item()  # eager work and a synchronisation
        graph.replay()
        torch.cuda.synchronize()
        out_eager, gx_eager = step()
        torch.cuda.synchronize()
        assert torch.equal(out_graph, out_eager) and torch.equal(gx_graph, gx_eager)


def test_eager_products_before_the_first_replay():
    """What a capture makes for a width that no product had before belongs to the graph: an eager product between
    the capture and its first replay, when none of it has run, makes its own."""
    data, _ = _make_data("copy", 64, True, 3, seed=4)
    data.to(DEV)
    plan = data.edge_index.plan()
    gen = torch.Generator(device=DEV)
    gen.manual_seed(10)
    narrow, wide = (torch.randn(data.vertex_cnt, F, device=DEV, generator=gen) for F in (20, 250))
    plan.forward(narrow), plan.backward(narrow)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out_graph, gx_graph = plan.forward(wide), plan.backward(wide)
    out_eager, gx_eager = plan.forward(wide), plan.backward(wide)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out_graph, out_eager) and torch.equal(gx_graph, gx_eager)
        assert torch.equal(plan.forward(wide), out_eager)


def test_first_products_of_a_plan_under_capture():
    """A plan whose first products are recorded: row numbers and run tables made on the way are the graph's too, so eager
    products (AUTO and the plain runs) between the capture and its first replay make their own."""
    data, _ = _make_data("copy", 64, True, 3, seed=4)
    data.to(DEV)
    plan = data.edge_index.plan()
    gen = torch.Generator(device=DEV)
    gen.manual_seed(11)
    x = torch.randn(data.vertex_cnt, 40, device=DEV, generator=gen)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out_graph, gx_graph = plan.forward(x), plan.backward(x)
        plan.method = "nnz_schedule"
        plain_graph = plan.forward(x)
        plan.method = "auto"
    out_eager, gx_eager = plan.forward(x), plan.backward(x)
    plan.method = "nnz_schedule"
    plain_eager = plan.forward(x)
    plan.method = "auto"
    fresh = _make_data("copy", 64, True, 3, seed=4)[0].to(DEV)  # a plan that was never recorded
    assert torch.equal(fresh.edge_index.plan().forward(x), out_eager)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out_graph, out_eager) and torch.equal(gx_graph, gx_eager) and torch.equal(plain_graph, plain_eager)
        assert torch.equal(plan.forward(x), out_eager) and torch.equal(plan.backward(x), gx_eager)


def test_spmm_func_int64_api():
    """The reference's raw operator on int64 CSR tensors, all accepted method strings."""
    import compressgnn_runtime as rt
    from util import random_csr
    rng = np.random.default_rng(2)
    vlist, elist, value = random_csr(rng, 300, 200, 5.0, skew=True)
    row_len = np.repeat(np.diff(vlist), np.diff(vlist))
    value = (value * 0.3 / np.sqrt(np.maximum(row_len, 1))).astype(np.float32)  # sym-norm-like weights
    x = rng.standard_normal((200, 48)).astype(np.float32)
    want = oracle.spmm(vlist, elist, value, x)
    t = lambda a: torch.from_numpy(a).to(DEV)
    for method in ["rowbalance_rowcache", "nnzbalance_rowcache", "rowbalance_parreduce", "nnzbalance_seqreduce"]:
        out = rt.spmm_func(t(vlist), t(elist), t(value), t(x), method, None)
        assert_within(out.cpu().numpy(), want)
        acc = t(np.ones((300, 48), np.float32))
        ret = rt.spmm_func(t(vlist), t(elist), t(value), t(x), method, acc)
        assert ret.data_ptr() == acc.data_ptr()
        assert_within(acc.cpu().numpy(), want + 1)
    with pytest.raises(RuntimeError):
        rt.spmm_func(t(vlist), t(elist), t(value), t(x), "no_such_method", None)
    with pytest.raises(RuntimeError):
        rt.spmm_func(torch.from_numpy(vlist), torch.from_numpy(elist), torch.from_numpy(value),
                     torch.from_numpy(x), "rowbalance", None)


def test_cluster_reconstruct_layers():
    from CompressgnnCluster import Compressgnn_Cluster, Compressgnn_Cluster_Function, _Mean
    from CompressgnnReconstruct import Compressgnn_Reconstruct
    torch.manual_seed(26)
    reconstruct = Compressgnn_Reconstruct()
    idx = torch.tensor([1, 1, 3, 1, 3, 3], device=DEV)
    count = torch.bincount(idx, minlength=5).int()
    x = torch.randn(6, 5, device=DEV, dtype=torch.double, requires_grad=True)
    assert torch.autograd.gradcheck(lambda a: _Mean.apply(a, idx, count), (x,), eps=1e-6, atol=1e-5, rtol=1e-3)
    for dtype in [torch.float32, torch.float64]:
        for width in [1, 31, 33, 128, 602]:
            for relu in [None, 'relu']:
                reps = torch.randn(5, width, device=DEV, dtype=dtype, requires_grad=True)
                bias = torch.randn(width, device=DEV, dtype=dtype, requires_grad=True)
                out = reconstruct(reps, idx, bias=bias, activation=relu)
                ref = reps.index_select(0, idx) + bias
                if relu:
                    ref = ref.relu()
                torch.testing.assert_close(out, ref, atol=1e-5, rtol=1e-4)
                go = torch.randn_like(out)
                a = torch.autograd.grad(out, (reps, bias), go)
                b = torch.autograd.grad(ref, (reps, bias), go)
                torch.testing.assert_close(a[0], b[0], atol=1e-5, rtol=1e-4)
                torch.testing.assert_close(a[1], b[1], atol=1e-5, rtol=1e-4)
    # what the layer keeps for its backward pass: the index and one bit per element, never the rows
    reps = torch.randn(5, 100, device=DEV, requires_grad=True)
    kept = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: kept.append(t) or t, lambda t: t):
        out = reconstruct(reps, idx, activation='relu')
    assert sorted((tuple(t.shape), t.dtype) for t in kept) == [((6,), torch.int64), ((6, 4), torch.int32)]
    kept.clear()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: kept.append(t) or t, lambda t: t):
        out = reconstruct(reps, idx)
    assert [tuple(t.shape) for t in kept] == [(6,)]
    reps = torch.randn(5, 3, device=DEV, dtype=torch.double, requires_grad=True)
    bias = torch.full((3,), 2., device=DEV, dtype=torch.double, requires_grad=True)
    assert torch.autograd.gradcheck(lambda a, b: reconstruct(a, idx, b, 'relu'), (reps, bias), eps=1e-6,
                                    atol=1e-5, rtol=1e-3)

    def scatter_mean(x, index, groups):
        s = torch.zeros(groups, x.size(1), device=x.device, dtype=x.dtype).index_add_(0, index, x)
        c = torch.bincount(index, minlength=groups).clamp_min(1).to(x.dtype)
        return s / c[:, None]

    c = Compressgnn_Cluster(7, 4, device=DEV, refresh_interval=5)
    ptr = None
    for epoch in range(12):
        x = torch.randn(19, 7, device=DEV, requires_grad=True)
        out, index = c(x, epoch=epoch, cache_key='graph-A')
        assert c.last_refreshed == (epoch % 5 == 0)
        if epoch % 5:
            assert index.data_ptr() == ptr
        ptr = index.data_ptr()
        ref = scatter_mean(x, index, out.size(0))
        torch.testing.assert_close(out, ref, atol=1e-5, rtol=1e-4)
        torch.testing.assert_close(torch.autograd.grad(out.square().sum(), x)[0],
                                   torch.autograd.grad(ref.square().sum(), x)[0], atol=1e-5, rtol=1e-4)
    assert c.refresh_count == 3
    # two shared transforms, one reconstruction, all parameter gradients
    layers = torch.nn.Sequential(torch.nn.Linear(7, 9), torch.nn.ReLU(), torch.nn.Linear(9, 3)).to(DEV)
    x = torch.randn(19, 7, device=DEV, requires_grad=True)
    rep, ii = c(x, epoch=15)
    out = reconstruct(layers(rep), ii)
    ref = layers(scatter_mean(x, ii, rep.size(0))).index_select(0, ii)
    torch.testing.assert_close(out, ref, atol=1e-5, rtol=1e-4)
    params = [x] + list(layers.parameters())
    aa = torch.autograd.grad(out.square().sum(), params)
    bb = torch.autograd.grad(ref.square().sum(), params)
    for a, b in zip(aa, bb):
        torch.testing.assert_close(a, b, atol=1e-5, rtol=1e-4)
    # non-default stream
    x = torch.randn(67, 33, device=DEV)
    w = torch.randn(33, 8, device=DEV)
    import compressgnn_runtime as native
    ri, rc, ra = native.cluster_assign(x, w, 8, native.cluster_workspace(x, 8))
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        ii, cc, aa = native.cluster_assign(x, w, 8, native.cluster_workspace(x, 8))
        yy = native.cluster_mean(x, ii, cc)
    stream.synchronize()
    assert torch.equal(ii, ri) and torch.equal(cc, rc) and aa == ra
    torch.testing.assert_close(yy, scatter_mean(x, ri, ra + 1), atol=1e-5, rtol=1e-4)
    # legacy entry
    a = Compressgnn_Cluster(7, 4, device=DEV)
    x = torch.randn(10, 7, device=DEV, requires_grad=True)
    y, ii, active = Compressgnn_Cluster_Function.apply(x, a.random_vectors, 4, True)
    ref = scatter_mean(x, ii, active + 1)
    torch.testing.assert_close(y, ref, atol=1e-5, rtol=1e-4)
    torch.testing.assert_close(torch.autograd.grad(y.sum(), x)[0], torch.autograd.grad(ref.sum(), x)[0],
                               atol=1e-5, rtol=1e-4)
    with pytest.raises(RuntimeError):
        native.cluster_assign(x, torch.randn(7, 3, device=DEV), 4, native.cluster_workspace(x, 4))


def test_kpu_propagate_hops_and_cache():
    """KPUPropagate (layer/KPUPropagate.py:25-37 of the reference): K hops per call; with
    cached=True the first result is kept and later calls return it detached, whatever their
    arguments, until reset_cache()."""
    from KPropagate import KPropagate
    from KPUPropagate import KPUPropagate
    data, _ = _make_data("copy", 32, True, 3, seed=2)
    data.to(DEV)
    args = (data.edge_index, None, data.vertex_cnt, data.rule_cnt)
    x = data.x.detach().clone().requires_grad_()
    hop = KPropagate()
    two = hop(hop(x, *args), *args)
    g = torch.randn(two.shape, device=DEV, generator=torch.Generator(device=DEV).manual_seed(1))
    (gx_two,) = torch.autograd.grad(two, x, g)
    kpu = KPUPropagate(K=2)
    out = kpu(x, *args)
    (gx,) = torch.autograd.grad(out, x, g)
    assert torch.equal(out, two) and torch.equal(gx, gx_two)  # the same kernels in the same order
    assert out.requires_grad and "K=2" in repr(kpu)
    # one hop of K=1 is KPropagate, and K=3 is one more hop on top of K=2
    assert torch.equal(KPUPropagate(K=1)(x, *args), hop(x, *args))
    assert torch.equal(KPUPropagate(K=3)(x, *args), hop(two, *args))
    # against the oracle: two applications of the compressed chain
    fwd_blocks, _ = _np_blocks(data.edge_index)
    want = oracle.compress_spmm_forward(fwd_blocks, oracle.compress_spmm_forward(fwd_blocks, data.x.cpu().numpy()))
    assert_within(out.detach().cpu().numpy(), want)

    cached = KPUPropagate(K=2, cached=True)
    first = cached(x, *args)
    assert first.requires_grad and torch.equal(first, two)
    other = torch.randn_like(x)
    second = cached(other, *args)  # arguments are ignored while the cache is filled
    assert not second.requires_grad and second.data_ptr() == first.data_ptr() and torch.equal(second, two)
    third = cached(other, *args)
    assert third.data_ptr() == first.data_ptr() and not third.requires_grad
    cached.reset_cache()
    fresh = cached(other, *args)
    assert fresh.data_ptr() != first.data_ptr()
    assert torch.equal(fresh, hop(hop(other, *args), *args))
    # without the cache every call propagates its own input
    plain = KPUPropagate(K=2, cached=False)
    assert torch.equal(plain(other, *args), fresh) and torch.equal(plain(x, *args), two)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n,width,bits", [(1, 5, 0), (67, 33, 8), (5000, 100, 12), (257, 128, 16), (300, 7, 20)])
def test_cluster_forward_entry(dtype, n, width, bits):
    """compressgnn_runtime.cluster_forward (src/runtime/csrc/cluster/cluster.cpp:12-30 of the
    reference): int32 ids, 1-based and dense in code order, and the number of active buckets."""
    import compressgnn_runtime as rt
    rng = np.random.default_rng(31 * n + bits)
    x = rng.standard_normal((n, width)).astype(dtype)
    planes = rng.standard_normal((width, bits)).astype(dtype)
    want_ids, want_active, _ = oracle.lsh(x, planes, bits)
    ids, active = rt.cluster_forward(torch.from_numpy(x).to(DEV), torch.from_numpy(planes).to(DEV), bits)
    assert ids.dtype == torch.int32 and ids.shape == (n,) and ids.is_cuda
    assert active == want_active
    assert np.array_equal(ids.cpu().numpy(), np.asarray(want_ids).astype(np.int32))
    with pytest.raises(RuntimeError):
        rt.cluster_forward(torch.from_numpy(x).to(DEV), torch.from_numpy(planes).to(DEV), bits + 1)
    with pytest.raises(RuntimeError):
        rt.cluster_forward(torch.from_numpy(x), torch.from_numpy(planes), bits)  # CPU tensors


def test_cluster_operators_reject_bad_operands():
    """Every operand check raises RuntimeError (the reference's TORCH_CHECKs do); ids that name
    no cluster are reported instead of read (the reference traps in the kernel)."""
    import compressgnn_runtime as rt
    x = torch.randn(50, 8, device=DEV)
    planes = torch.randn(8, 4, device=DEV)
    ids, counts, active = rt.cluster_assign(x, planes, 4, rt.cluster_workspace(x, 4))
    groups = active + 1
    reps = rt.cluster_mean(x, ids, counts)
    bad_calls = [
        lambda: rt.cluster_workspace(x, 31),
        lambda: rt.cluster_workspace(x.to(torch.int32), 4),
        lambda: rt.cluster_assign(x, planes, 4, rt.cluster_workspace(x, 5)),       # workspace of another size
        lambda: rt.cluster_assign(x, planes, 4, rt.cluster_workspace(x, 4)[:2]),
        lambda: rt.cluster_assign(x, planes.double(), 4, rt.cluster_workspace(x, 4)),
        lambda: rt.cluster_assign(x.t(), planes, 4, rt.cluster_workspace(x, 4)),  # not contiguous
        lambda: rt.cluster_mean(x, ids.to(torch.int32), counts),
        lambda: rt.cluster_mean(x, ids[:-1], counts),
        lambda: rt.cluster_mean(x, ids, counts.to(torch.int64)),
        lambda: rt.cluster_mean(x, ids.cpu(), counts),
        lambda: rt.cluster_mean_backward(reps[:-1], ids, counts),
        lambda: rt.cluster_reconstruct(reps, ids, torch.zeros(7, device=DEV), False),
        lambda: rt.cluster_reconstruct(reps, ids, torch.zeros(8, device=DEV, dtype=torch.double), False),
        lambda: rt.cluster_reconstruct_backward(torch.zeros(50, 8, device=DEV), ids, torch.zeros(50, 9, device=DEV),
                                                groups, True),
        lambda: rt.cluster_reconstruct_signs(reps, ids, torch.zeros(7, device=DEV)),
        lambda: rt.cluster_reconstruct_backward_signs(torch.zeros(50, 8, device=DEV), ids,
                                                      torch.zeros(50, 2, device=DEV, dtype=torch.int32), groups),
        lambda: rt.cluster_reconstruct_backward_signs(torch.zeros(50, 8, device=DEV), ids,
                                                      torch.zeros(50, 1, device=DEV), groups),  # words are int32
        lambda: rt.cluster_members(ids, 0),
    ]
    for k, call in enumerate(bad_calls):
        with pytest.raises(RuntimeError):
            call()
            raise AssertionError("bad call %d was accepted" % k)
    # ids beyond the representatives: an error, never an access outside the arrays
    beyond = ids.clone()
    beyond[7] = groups + 3
    negative = ids.clone()
    negative[0] = -1
    for index in (beyond, negative):
        with pytest.raises(RuntimeError, match="outside"):
            rt.cluster_reconstruct(reps, index, None, False)
        with pytest.raises(RuntimeError, match="outside"):
            rt.cluster_reconstruct_signs(reps, index, None)
        with pytest.raises(RuntimeError, match="outside"):
            rt.cluster_reconstruct_backward_signs(torch.zeros(50, 8, device=DEV), index,
                                                  torch.zeros(50, 1, device=DEV, dtype=torch.int32), groups)
        with pytest.raises(RuntimeError, match="outside"):
            rt.cluster_mean_backward(reps, index, counts)
        with pytest.raises(RuntimeError, match="outside"):
            rt.cluster_members(index, groups)
        with pytest.raises(RuntimeError, match="outside"):
            rt.cluster_mean(x, index, counts)  # builds the member lists itself
        with pytest.raises(RuntimeError, match="outside"):
            rt.cluster_reconstruct_backward(torch.zeros(50, 8, device=DEV), index, torch.ones(50, 8, device=DEV),
                                            groups, True)
    # the device is fine afterwards and the good calls still give the same results
    torch.cuda.synchronize()
    assert torch.equal(rt.cluster_mean(x, ids, counts), reps)
    from CompressgnnReconstruct import Compressgnn_Reconstruct
    with pytest.raises(RuntimeError, match="outside"):
        Compressgnn_Reconstruct()(reps, beyond)


def test_reference_method_strings_are_hints():
    """The reference's layers ask for "rowbalance_rowcache" on every block of 1e6 non-zeros and
    width >= 64 (layer/CompressgnnSPMM.py:14-19,34,38), whatever its rows look like.  On a block
    with power-law rows the string must not force a lane group per row: same result as "auto"
    (bit for bit: the same schedule runs), within tolerance of the oracle, and no slower than a
    small multiple of "auto"."""
    import compressgnn_runtime as rt
    rng = np.random.default_rng(8)
    rows, cols, F = 60000, 60000, 64
    lens = np.minimum((rng.pareto(1.1, rows) * 3).astype(np.int64) + 1, 40000)
    lens[rng.integers(0, rows, 3)] = 60000  # three hub rows
    vlist = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    elist = rng.integers(0, cols, int(vlist[-1])).astype(np.int64)
    value = (rng.standard_normal(len(elist)) * 0.3 / np.sqrt(np.repeat(lens, lens))).astype(np.float32)
    x = rng.standard_normal((cols, F)).astype(np.float32)
    t = lambda a: torch.from_numpy(a).to(DEV)
    tv, te, tw, tx = t(vlist), t(elist), t(value), t(x)
    auto = rt.spmm_func(tv, te, tw, tx, "auto", None)
    hinted = rt.spmm_func(tv, te, tw, tx, "rowbalance_rowcache", None)
    assert torch.equal(auto, hinted)
    want = oracle.spmm(vlist, elist, value, x, None, 8)
    # rows of up to 60,000 entries: the sequential fp32 sum is itself several 1e-6 from the exact
    # value, so the kernel is held to being no further from float64 than the oracle is
    truth = np.zeros((rows, F))
    np.add.at(truth, np.repeat(np.arange(rows), lens), value[:, None].astype(np.float64) * x[elist])
    assert_no_less_accurate(hinted.cpu().numpy(), want, truth, factor=1.5)
    assert_within(hinted.cpu().numpy(), want, rtol=1e-4, atol=1e-5)

    def timed(method):
        rt.spmm_func(tv, te, tw, tx, method, None)
        torch.cuda.synchronize()
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(5):
            rt.spmm_func(tv, te, tw, tx, method, None)
        b.record()
        torch.cuda.synchronize()
        return a.elapsed_time(b) / 5

    t_auto, t_hint = timed("auto"), timed("rowbalance_rowcache")
    assert t_hint <= 1.5 * t_auto + 0.05, (t_hint, t_auto)
    # a forced row schedule stays available under this build's own name, bit-exact with the oracle
    forced = rt.DeviceCsr(tv, te, tw, rows, cols, torch.device(DEV)).spmm(tx, None, "row_schedule")
    assert np.array_equal(forced.cpu().numpy(), want)


def test_propagation_from_representatives_equals_propagation_of_the_written_rows():
    """GatheredPropagate(small, index, graph) against KPropagate on small[index]: the same bits,
    forward and gradient, for an assignment of Compressgnn_Cluster and for an index from
    elsewhere, folded and launch-per-level plans; an id that names no cluster is refused; a new
    assignment is noticed."""
    from CompressgnnCluster import Compressgnn_Cluster
    from GatheredPropagate import GatheredPropagate
    from KPropagate import KPropagate
    for fold in (True, False):
        data, _ = _make_data("copy", 64, True, 3, seed=6)
        data.to(DEV)
        graph = data.edge_index
        graph.fold_levels = fold
        V, F = data.vertex_cnt, 64
        torch.manual_seed(3)
        cluster = Compressgnn_Cluster(in_feature=F, param_H=7, training=True, cache=False).to(DEV)
        reps, index = cluster(data.x)
        C = reps.size(0)
        g = torch.randn(V, F, device=DEV)
        for idx in (index, torch.randint(0, C, (V,), device=DEV)):
            small = torch.randn(C, F, device=DEV, requires_grad=True)
            out = GatheredPropagate()(small.relu(), idx, graph)
            (d_small,) = torch.autograd.grad(out, small, g)
            small2 = small.detach().clone().requires_grad_()
            rows = small2.relu().index_select(0, idx)
            want = KPropagate()(rows, graph, None, data.vertex_cnt, data.rule_cnt)
            (d_want,) = torch.autograd.grad(want, small2, g)
            assert torch.equal(out, want)
            # the dense path sums a cluster's gradient through index_select's backward (atomics in
            # torch); the member-list sum has a fixed order
            ref = torch.zeros(C, F, dtype=torch.float64, device=DEV).index_add_(
                0, idx, graph.plan().backward(g).double()) * (small.detach() > 0)
            assert_within(d_small.cpu().numpy(), ref.cpu().numpy(), rtol=1e-5, atol=1e-6)
            assert_within(d_want.cpu().numpy(), ref.cpu().numpy(), rtol=1e-4, atol=1e-5)
        # a refreshed assignment (another tensor) is composed anew
        reps_b, index_b = cluster(data.x * 1.5 + 0.1)
        small = torch.randn(reps_b.size(0), F, device=DEV)
        assert torch.equal(GatheredPropagate()(small, index_b, graph),
                           KPropagate()(small.index_select(0, index_b), graph, None, data.vertex_cnt, data.rule_cnt))
        bad = index_b.clone()
        bad[5] = reps_b.size(0) + 3
        with pytest.raises(RuntimeError, match="outside"):
            GatheredPropagate()(small, bad, graph)
        with pytest.raises(ValueError):
            GatheredPropagate()(small, index_b[:-1], graph)
    # a graph without rules: the rule stage has nothing to do
    data, _ = _make_data("chung_lu", 32, True, 10 ** 6, seed=2)
    assert data.rule_cnt == 0
    data.to(DEV)
    idx = torch.randint(0, 50, (data.vertex_cnt,), device=DEV)
    small = torch.randn(50, 32, device=DEV)
    assert torch.equal(GatheredPropagate()(small, idx, data.edge_index),
                       KPropagate()(small.index_select(0, idx), data.edge_index, None, data.vertex_cnt, data.rule_cnt))


def test_a_later_plan_applies_the_orders_the_first_one_found(tmp_path, monkeypatch):
    """The locality orders of the two vertex stages depend on the blocks alone: the graph keeps them,
    a dataset saved with torch.save carries them, and a plan built later (after loading, after
    another to(device)) does not search again -- the search routine is made to raise here -- and
    propagates to the same bits, forward and backward."""
    import compress_graph
    data, _ = _make_data("copy", 48, True, 3, seed=6)
    assert data.edge_index._stage_orders is None
    data.to(DEV)
    graph = data.edge_index
    plan = graph.plan()
    V = data.vertex_cnt
    for order in graph._stage_orders.values():
        assert order.dtype == np.int32 and np.array_equal(np.sort(order), np.arange(V))
    gen = torch.Generator(device=DEV).manual_seed(3)
    x = torch.randn(V, 48, device=DEV, generator=gen)
    g = torch.randn(V, 48, device=DEV, generator=gen)
    out, gx = plan.forward(x), plan.backward(g)
    path = str(tmp_path / "prepared.pt")
    torch.save(data, path)  # this test's own file
    loaded = torch.load(path, weights_only=False)

    def no_search(*_):
        raise AssertionError("the locality order was searched for again")

    monkeypatch.setattr(compress_graph, "csr_locality_order", no_search)
    loaded.to(DEV)
    again = loaded.edge_index.plan()
    assert torch.equal(again.forward(x), out) and torch.equal(again.backward(g), gx)
    graph.to(DEV)  # drops the plan, keeps the orders
    assert graph._plan is None
    once_more = graph.plan()
    assert torch.equal(once_more.forward(x), out) and torch.equal(once_more.backward(g), gx)


def test_uncompressed_hop_over_an_edge_tensor():
    """Propagate.propagate(edge_index, x, edge_weight) with a [2, E] edge tensor
    (layer/CompressgnnPropagation.py:50-60, edge-tensor branch): out[dst] += w * x[src] in edge
    order per destination, i.e. bit-equal to the oracle's sequential scatter-add where a
    destination takes the row schedule; the gradient is the transposed sum; without weights every
    edge counts 1; duplicate edges and vertices without edges included."""
    import prep_oracle
    from KPropagate import KPropagate
    rng = np.random.default_rng(17)
    V, E, F = 3000, 26000, 40
    src = rng.integers(0, V, E)
    dst = rng.integers(0, V - 200, E)  # the last 200 vertices receive nothing
    src[:50], dst[:50] = src[50:100], dst[50:100]  # duplicate edges
    w = (rng.standard_normal(E) * 0.3).astype(np.float32)
    x_np = rng.standard_normal((V, F)).astype(np.float32)
    edges = np.vstack((src, dst)).astype(np.int64)
    want = prep_oracle.coo_propagate(x_np, [edges], [w], V, 0)
    g_np = rng.standard_normal((V, F)).astype(np.float32)
    want_gx = np.zeros_like(x_np)
    np.add.at(want_gx, src, w.reshape(-1, 1) * g_np[dst])
    prop = KPropagate()
    x = torch.from_numpy(x_np).to(DEV).requires_grad_()
    e_t, w_t = torch.from_numpy(edges).to(DEV), torch.from_numpy(w).to(DEV)
    out = prop.propagate(e_t, x, w_t)
    (gx,) = torch.autograd.grad(out, x, torch.from_numpy(g_np).to(DEV))
    assert_within(out.detach().cpu().numpy(), want)
    assert_within(gx.cpu().numpy(), want_gx, rtol=1e-5, atol=2e-6)
    assert not out[V - 200:].any()
    ones = prop.propagate(e_t, x)
    assert_within(ones.detach().cpu().numpy(), prep_oracle.coo_propagate(x_np, [edges], [np.ones(E, np.float32)], V, 0))
    with pytest.raises(TypeError):
        prop.propagate([e_t], x, w_t)


@pytest.mark.parametrize("weights", [True, False])
@pytest.mark.parametrize("kind", ["chain", "deep_chain", "no_rules", "used_before_complete", "vertex_source_late"])
def test_phase_lists_of_every_shape(kind, weights):
    """Phase lists that are a compressed chain (with and without levels, too deep to fold, without rules) and lists
    that are not (a rule reached after it was a source; a vertex as a source of a later phase), forward and
    gradient against the gather + scatter-add loop in float64."""
    from CooPhases import CooPhasePlan, coo_propagate
    rng = np.random.default_rng(3)
    V, R, F = 90, 0 if kind == "no_rules" else 40, 20
    vert = lambda n: rng.integers(0, V, n)
    lo = lambda a, b, n: V + rng.integers(a, b, n)
    phases = [(vert(400), np.concatenate([vert(300), lo(0, 10, 100) if R else vert(100)]))]
    if kind == "chain":
        phases += [(lo(0, 10, 60), vert(60))]
    if kind in ("deep_chain", "used_before_complete", "vertex_source_late"):
        steps = 20 if kind == "deep_chain" else 3
        for k in range(steps):  # rules of stage k feed stage k + 1 (two rules a stage) and vertices
            a = 0 if k == 0 else 10 + (k - 1)
            b = 10 if k == 0 else a + 1
            phases += [(np.concatenate([lo(a, b, 8), lo(a, b, 12)]), np.concatenate([lo(10 + k, 11 + k, 8), vert(12)]))]
    if kind == "used_before_complete":
        phases += [(lo(11, 12, 9), lo(0, 10, 9))]
    if kind == "vertex_source_late":
        phases += [(vert(9), vert(9))]
    w = [rng.standard_normal(len(s)).astype(np.float32) if weights else None for s, _ in phases]
    t = lambda a: torch.from_numpy(a).to(DEV)
    edges = [torch.stack([t(s), t(d)]) for s, d in phases]
    plan = CooPhasePlan(edges, [t(a) for a in w] if weights else None, V, R)
    assert (plan.chain is not None) == (kind in ("chain", "deep_chain", "no_rules"))
    x, g = rng.standard_normal((V, F)).astype(np.float32), rng.standard_normal((V, F)).astype(np.float32)
    full = np.zeros((V + R, F))
    for k, (s, d) in enumerate(phases):
        source = x.astype(np.float64) if k == 0 else full.copy()
        np.add.at(full, d, (1.0 if w[k] is None else w[k][:, None].astype(np.float64)) * source[s])
    back = np.concatenate([g.astype(np.float64), np.zeros((R, F))])
    gx = np.zeros((V, F))
    for k in range(len(phases) - 1, -1, -1):
        s, d = phases[k]
        move = (1.0 if w[k] is None else w[k][:, None].astype(np.float64)) * back[d]
        np.add.at(gx if k == 0 else back, s, move)
    X = t(x).requires_grad_()
    out = coo_propagate(plan, X)
    (got,) = torch.autograd.grad(out, X, t(g))
    np.testing.assert_allclose(out.detach().cpu().numpy(), full[:V], rtol=1e-4, atol=1e-4 * np.abs(full[:V]).max())
    np.testing.assert_allclose(got.cpu().numpy(), gx, rtol=1e-4, atol=1e-4 * np.abs(gx).max())


@pytest.mark.parametrize("shape", ["one_row", "no_long_rows", "hubs_first", "empty_tail", "empty_head", "places_full", "mixed"])
@pytest.mark.parametrize("accumulate", [False, True])
def test_spmm_func_on_blocks_of_every_shape(shape, accumulate):
    """The operator on int64 tensors narrows its block in stretches of 2,048 rows and entries: rows that end or begin
    with a stretch, rows over several stretches, thousands of empty rows in front, behind and between; against
    float64, and bit for bit where a row has at most 64 entries."""
    import compressgnn_runtime as rt
    rng = np.random.default_rng(17)
    lens = {"one_row": [5000], "no_long_rows": rng.integers(0, 9, 3000), "hubs_first": [9000, 2048, 2047, 2049] + [1] * 500,
            "empty_tail": [3, 70, 2] + [0] * 9000, "empty_head": [0] * 9000 + [1, 3000, 64, 65],
            "places_full": [2047, 2047, 2046, 0, 2047, 1023, 1023, 0, 0],
            "mixed": np.where(rng.random(4000) < 0.6, 0, rng.integers(0, 200, 4000))}[shape]
    lens = np.asarray(lens, np.int64)
    vlist = np.concatenate([[0], np.cumsum(lens)])
    cols, F = 700, 20
    elist = rng.integers(0, cols, int(vlist[-1]))
    value = (rng.standard_normal(len(elist)) * 0.3 / np.sqrt(np.maximum(np.repeat(lens, lens), 1))).astype(np.float32)
    x = rng.standard_normal((cols, F)).astype(np.float32)
    out0 = rng.standard_normal((len(lens), F)).astype(np.float32) if accumulate else np.zeros((len(lens), F), np.float32)
    want = out0.astype(np.float64)
    np.add.at(want, np.repeat(np.arange(len(lens)), lens), value[:, None].astype(np.float64) * x[elist])
    t = lambda a: torch.from_numpy(a).to(DEV)
    for _ in range(2):
        got = rt.spmm_func(t(vlist), t(elist), t(value), t(x), "auto", t(out0.copy()) if accumulate else None).cpu().numpy()
        assert_within(got, want, rtol=1e-5, atol=2e-5)
    short = lens <= 64
    assert np.array_equal(got[short], oracle.spmm(vlist, elist, value, x, out0.copy())[short])


@pytest.mark.parametrize("rows, nnz", [(1, 5), (63, 1), (64, 4033), (65, 4096 - 65), (4097, 9999), (400000, 1172864), (400000, 1172865),
                                       (1572000, 1000)])
def test_spmm_func_of_any_length(rows, nnz):
    """Blocks on both sides of the rows and entries that a workgroup and its search for them take, with a hub, a stretch of
    empty rows and an empty last row.  Whole numbers, so every order of the sums gives the same bits."""
    import compressgnn_runtime as rt
    rng = np.random.default_rng(rows + nnz)
    ends = np.sort(np.concatenate([rng.integers(0, nnz + 1, rows - rows // 3), np.full(rows // 3, nnz // 2)]))
    vlist = np.concatenate([[0], ends]).astype(np.int64)
    vlist[-2:] = nnz
    vlist[0] = 0
    elist = rng.integers(0, 500, nnz).astype(np.int64)
    value = rng.integers(-3, 4, nnz).astype(np.float32)
    x = rng.integers(-3, 4, (500, 4)).astype(np.float32)
    sums = np.concatenate([np.zeros((1, 4)), np.cumsum(value[:, None] * x[elist].astype(np.float64), 0)])
    want = (sums[vlist[1:]] - sums[vlist[:-1]]).astype(np.float32)
    t = lambda a: torch.from_numpy(a).to(DEV)
    for _ in range(2):
        assert np.array_equal(rt.spmm_func(t(vlist), t(elist), t(value), t(x), "auto", None).cpu().numpy(), want)


@pytest.mark.parametrize("method", ["auto", "row_schedule", "nnz_schedule"])
@pytest.mark.parametrize("hubs", [False, True])
@pytest.mark.parametrize("rows", [(0, 3000), (1, 3000), (0, 2999), (1234, 1235), (700, 2900)])
def test_spmm_func_on_a_slice_of_the_rows(rows, hubs, method):
    """Row pointers sliced out of a larger block, with all its entries, and lists padded behind the last row: the rows
    of the whole product, bit for bit where a row is never divided.  Entries outside the rows are NaN: none is used."""
    import compressgnn_runtime as rt
    rng = np.random.default_rng(23)
    lens = rng.integers(0, 9, 3000)
    if hubs:
        lens[::500] = 3000
    vlist = np.concatenate([[0], np.cumsum(lens)])
    cols, F = 700, 20
    elist = rng.integers(0, cols, int(vlist[-1]))
    value = (rng.standard_normal(len(elist)) * 0.3 / np.sqrt(np.maximum(np.repeat(lens, lens), 1))).astype(np.float32)
    x = rng.standard_normal((cols, F)).astype(np.float32)
    t = lambda a: torch.from_numpy(a).to(DEV)
    whole = np.zeros((len(lens), F))
    np.add.at(whole, np.repeat(np.arange(len(lens)), lens), value[:, None].astype(np.float64) * x[elist])
    sequential = oracle.spmm(vlist, elist, value, x)
    a, b = rows
    outside = np.ones(len(elist) + 777, bool)
    outside[vlist[a]:vlist[b]] = False
    padded = np.concatenate([value, np.zeros(777, np.float32)])
    padded[outside] = np.nan
    args = t(vlist[a:b + 1].copy()), t(np.concatenate([elist, np.zeros(777, np.int64)])), t(padded)
    got = rt.spmm_func(*args, t(x), method, None).cpu().numpy()
    assert_within(got, whole[a:b], rtol=1e-5, atol=2e-5)
    short = lens[a:b] <= 64
    assert np.array_equal(got[short], sequential[a:b][short])
    added = rt.spmm_func(*args, t(x), method, torch.ones(b - a, F, device=DEV)).cpu().numpy()
    assert_within(added, whole[a:b] + 1, rtol=1e-5, atol=2e-5)
    wide = rt.spmm_func(args[0], args[1], args[2].double(), t(x).double(), method, None).cpu().numpy()
    np.testing.assert_allclose(wide, whole[a:b], rtol=1e-12, atol=1e-12)


def test_products_of_one_plan_from_several_threads():
    """Forward in one thread, forward and gradient (which runs on the engine's thread) in others, all over one plan and one
    stream, at widths that make each product ask for other scratch, counters and tables: every result is that of a
    program with one thread, and the timer keeps its records whole."""
    import threading
    from KPropagate import KPropagate
    data, _ = _make_data("copy", 8, True, 3, seed=4)
    data.to(DEV)
    graph, hop = data.edge_index, KPropagate()
    plan = graph.plan()
    plan.timed_stages = ["bwd.final"]
    gen = torch.Generator(device=DEV)
    gen.manual_seed(12)
    widths = [5, 250, 16, 130, 33, 64]
    inputs = {F: torch.randn(data.vertex_cnt, F, device=DEV, generator=gen) for F in widths}

    def step(x, F):
        x = x.detach().requires_grad_()
        out = hop(x, graph, None, data.vertex_cnt, data.rule_cnt)
        return out.detach(), torch.autograd.grad(out, x, inputs[F])[0]

    failures, rounds = [], 12
    results = [[] for _ in range(3)]

    def work(k):
        try:
            for r in range(rounds):
                F = widths[(r + 2 * k) % len(widths)]
                results[k].append((F,) + (step(inputs[F], F) if k else (plan.forward(inputs[F]),)))
        except Exception as e:  # reported by the test's own thread
            failures.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures, failures
    times = plan.take_stage_times()
    assert len(times) == 2 * rounds and all(name == "bwd.final" and ms > 0 for name, ms in times)
    plan.timed_stages = []
    for k in range(3):
        for F, *got in results[k]:
            want = step(inputs[F], F)
            assert all(torch.equal(a, b) for a, b in zip(got, want))


def _steps_of_every_layer():
    """(name, function of one tensor, rows, width) of each layer's differentiable step."""
    from CompressgnnCluster import Compressgnn_Cluster
    from CompressgnnReconstruct import Compressgnn_Reconstruct
    from KPropagate import KPropagate
    data, _ = _make_data("copy", 8, True, 3, seed=4)
    data.to(DEV)
    V, hop = data.vertex_cnt, KPropagate()
    edges = torch.randint(0, V, (2, 4 * V), device=DEV)
    torch.manual_seed(6)
    fresh = Compressgnn_Cluster(12, 5, training=True, device=DEV, cache=False)
    held = Compressgnn_Cluster(12, 5, training=True, device=DEV, refresh_interval=5)
    with torch.no_grad():
        held(torch.randn(V, 12, device=DEV), epoch=0)
    groups = held.active_bucket + 1
    bias = torch.randn(12, device=DEV)
    return [("csr", lambda x: hop(x, data.edge_index, None, V, data.rule_cnt), V, 12),
            ("coo", lambda x: hop.propagate(edges, x), V, 12),
            ("cluster_fresh", lambda x: fresh(x)[0], V, 12),
            ("cluster_held", lambda x: held(x, epoch=1)[0], V, 12),
            ("reconstruct", lambda x: Compressgnn_Reconstruct()(x, held.vertex_index, bias, "relu"), groups, 12)]


@pytest.mark.filterwarnings("ignore")
def test_steps_where_a_native_one_would_be_lost():
    """torch.jit.trace records a layer as an operation on its input; tangents and torch.func transforms are refused (no
    layer has rules for them) and never dropped; all but the propagation of a CompressGraph refuse a second differentiation."""
    import torch.autograd.forward_ad as forward_mode
    import compressgnn_runtime as rt
    for name, step, rows, width in _steps_of_every_layer():
        x, y = (torch.randn(rows, width, device=DEV) for _ in range(2))
        with forward_mode.dual_level():
            with pytest.raises(NotImplementedError):
                step(forward_mode.make_dual(x, y))
        with pytest.raises(RuntimeError):
            torch.func.grad(lambda t: step(t).sum())(x)
        with pytest.raises(RuntimeError):
            torch.func.vmap(step)(torch.stack([x, y]))
        if name == "cluster_fresh":  # a trace cannot hold an assignment that is made anew
            with pytest.raises(RuntimeError):
                torch.jit.trace(step, (x,), check_trace=False)
        else:
            traced = torch.jit.trace(step, (x,), check_trace=False)
            assert torch.equal(traced(x), step(x)) and torch.equal(traced(y), step(y)), name
        z = x.clone().requires_grad_()
        first, = torch.autograd.grad(step(z).square().sum(), z, create_graph=True)
        again = (first * y).sum() + (z * y).sum()
        if name == "csr":  # no second-order term, as Compressgnn_SPMM_Function has none
            again.backward()
            assert torch.equal(z.grad, y)
        else:
            with pytest.raises(RuntimeError, match="twice"):
                again.backward()
    with forward_mode.dual_level():
        dual = forward_mode.make_dual(x, y)
        assert rt.reconstruct(dual, torch.zeros(5, dtype=torch.int64, device=DEV), None, False) is None


@pytest.mark.parametrize("kind", ["chain", "levels", "no_rules", "vertex_source_late"])
def test_edge_lists_of_either_precision_and_from_several_devices(kind):
    """Without weights the features may be float64, in lists that run as a chain and in others; with weights (32 bits)
    they may not.  Edges and weights may lie elsewhere than the first phase; a weight per edge is asked for phase by phase."""
    from CooPhases import CooPhasePlan, coo_propagate
    rng = np.random.default_rng(8)
    V, R, F = 300, 0 if kind == "no_rules" else 40, 11
    vert = lambda n: rng.integers(0, V, n)
    phases = [np.stack([vert(900), np.concatenate([vert(700), V + rng.integers(0, 10, 200) if R else vert(200)])])]
    if kind == "levels":
        phases += [np.stack([V + rng.integers(0, 10, 10), V + rng.integers(10, 20, 10)])]
    if R:
        phases += [np.stack([V + rng.integers(10 if kind == "levels" else 0, 20 if kind == "levels" else 10, 60), vert(60)])]
    if kind == "vertex_source_late":
        phases += [np.stack([vert(9), vert(9)])]
    x, g = rng.standard_normal((V, F)), rng.standard_normal((V, F))
    full, back, gx = np.zeros((V + R, F)), np.concatenate([g, np.zeros((R, F))]), np.zeros((V, F))
    for k, (s, d) in enumerate(phases):
        source = x if k == 0 else full.copy()
        np.add.at(full, d, source[s])
    for k in range(len(phases) - 1, -1, -1):
        s, d = phases[k]
        moved = back[d]
        np.add.at(gx if k == 0 else back, s, moved)
    edges = [torch.from_numpy(p).to(DEV if k == 0 else "cpu") for k, p in enumerate(phases)]
    plan = CooPhasePlan(edges, None, V, R)
    assert (plan.chain is not None) == (kind != "vertex_source_late")
    for dtype, tol in ((torch.float64, 1e-12), (torch.float32, 1e-4), (torch.float64, 1e-12)):
        X = torch.from_numpy(x).to(DEV, dtype).requires_grad_()
        out = coo_propagate(plan, X)
        (got,) = torch.autograd.grad(out, X, torch.from_numpy(g).to(DEV, dtype))
        assert out.dtype == got.dtype == dtype
        np.testing.assert_allclose(out.detach().cpu().numpy(), full[:V], rtol=tol, atol=tol * np.abs(full).max())
        np.testing.assert_allclose(got.cpu().numpy(), gx, rtol=tol, atol=tol * np.abs(gx).max())
    with pytest.raises(RuntimeError):
        coo_propagate(plan, X.detach().half())
    ones = [torch.ones(p.shape[1], dtype=torch.float64) for p in phases]
    weighted = CooPhasePlan(edges, ones, V, R)
    np.testing.assert_allclose(coo_propagate(weighted, X.detach().float()).cpu().numpy(), full[:V], rtol=1e-4,
                               atol=1e-4 * np.abs(full).max())
    with pytest.raises(RuntimeError):
        coo_propagate(weighted, X.detach())
    for wrong in ([ones[0][:, None]] + ones[1:], [ones[0][:-1]] + [torch.ones(len(w) + 1) for w in ones[1:]]):
        with pytest.raises(ValueError):
            CooPhasePlan(edges, wrong, V, R)


@pytest.mark.parametrize("call", ["assignment", "sampler"])
def test_other_threads_run_while_a_call_waits_for_the_stream(call):
    """The host read of an assignment and of a sampled batch stands behind what the stream has still to do; the other
    threads of the interpreter go on meanwhile."""
    import threading
    import time
    import compressgnn_runtime as rt
    import compressgnn_sample as sampler
    gen = torch.Generator(device=DEV)
    gen.manual_seed(13)
    if call == "assignment":
        x, planes = (torch.randn(n, m, device=DEV, generator=gen) for n, m in ((40000, 32), (32, 12)))
        run = lambda: rt.cluster_assign_members(x, planes, 12)[0]
    else:
        ptr = torch.arange(0, 3 * 5000 + 1, 3, device=DEV)
        col, seeds = (torch.randint(0, 5000, (n,), device=DEV, generator=gen) for n in (15000, 64))
        run = lambda: sampler.neighbor_sample_ori_impl(ptr, col, seeds, [5, 5], seed=2)[0]
    a = torch.randn(8192, 8192, device=DEV, generator=gen)
    out = torch.empty_like(a)
    want = run().clone()
    torch.mm(a, a, out=out)
    torch.cuda.synchronize()
    stamps, stop = [], threading.Event()

    def tick():
        while not stop.is_set():
            stamps.append(time.perf_counter())
            time.sleep(0.0005)

    ticker = threading.Thread(target=tick)
    ticker.start()
    try:
        time.sleep(0.02)
        for _ in range(16):  # 1.1 TFLOP each
            torch.mm(a, a, out=out)
        begin = time.perf_counter()
        got = run()
        end = time.perf_counter()
        time.sleep(0.02)
    finally:
        stop.set()
        ticker.join()
    assert torch.equal(got, want)
    assert end - begin > 0.03, "the stream was not busy"
    inside = [begin] + [t for t in stamps if begin < t < end] + [end]
    longest = max(later - earlier for earlier, later in zip(inside, inside[1:]))
    assert longest < 0.5 * (end - begin)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("width", [1, 3, 16, 33, 64, 130, 200, 512, 520, 1030])
def test_products_of_int64_arrays_of_every_shape(width, dtype):
    """spmm_func looks for the rows of a workgroup's entries itself: numbers of rows around a step of the search and around what
    the workgroup reads of them at once, rows without entries in front, between and behind, rows at the lengths that are moved
    or divided, hubs over many workgroups, slices and padded lists.  Whole numbers: the sums are exact in any order."""
    import compressgnn_runtime as rt
    rng = np.random.default_rng(width)
    lengths = [[5], [0, 0, 3], [0] * 300 + [70] + [0] * 700, [1] * 129, [64] * 128, [65] * 64, [63, 64, 65, 0, 31, 32, 33] * 40,
               [0, 1] * 3000, [5000], [1, 3000, 1, 0, 700] * 9, rng.integers(0, 40, 255).tolist(), rng.integers(0, 3, 8200).tolist(),
               (rng.pareto(1.2, 4097) * 3).astype(int).clip(0, 4000).tolist(), rng.integers(0, 20, 16385).tolist()]
    for lens in lengths:
        cols = 500
        v = np.concatenate([[0], np.cumsum(lens)])
        pad = int(rng.integers(0, 3)) * 777  # entries that no row holds
        first = int(rng.integers(0, 2)) * 130
        e = torch.from_numpy(rng.integers(0, cols, first + v[-1] + pad)).to(DEV)
        ptr = torch.from_numpy(v + first).to(DEV)
        w = torch.from_numpy(rng.integers(-3, 4, len(e))).to(DEV).to(dtype)
        x = torch.from_numpy(rng.integers(-8, 9, (cols, width))).to(DEV).to(dtype)
        rows = torch.repeat_interleave(torch.arange(len(lens), device=DEV), torch.tensor(lens, device=DEV))
        inside = slice(first, first + int(v[-1]))
        want = torch.zeros(len(lens), width, device=DEV, dtype=dtype)
        for at in range(0, int(v[-1]), 1 << 14):  # in parts: no array of all products
            part = slice(inside.start + at, min(inside.stop, inside.start + at + (1 << 14)))
            want.index_add_(0, rows[at:at + (1 << 14)], x[e[part]] * w[part, None])
        w[:first], w[inside.stop:] = float("nan"), float("nan")
        for _ in range(2):
            assert torch.equal(rt.spmm_func(ptr, e, w, x, "auto", None), want)
        base = torch.from_numpy(rng.integers(-9, 9, (len(lens), width))).to(DEV).to(dtype)
        assert torch.equal(rt.spmm_func(ptr, e, w, x, "auto", base.clone()), base + want)
    nothing = torch.full((1000,), 40, device=DEV, dtype=torch.int64)  # a slice whose rows are all empty
    assert not rt.spmm_func(nothing, e, w, x, "auto", None).any()


def rows_with_entries(rows, taken, rng, cols=300):
    """Row pointers and columns of a block: taken = {row: entries}, all other rows without entries."""
    lens = np.zeros(rows, np.int64)
    for row, n in taken.items():
        lens[row] = n
    v = np.concatenate([[0], np.cumsum(lens)])
    return lens, torch.from_numpy(v).to(DEV), torch.from_numpy(rng.integers(0, cols, int(v[-1]))).to(DEV)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("width", [1, 8, 33, 200, 257, 512, 602])
def test_products_of_int64_arrays_with_stretches_of_empty_rows(width, dtype):
    """Rows without entries between those of one workgroup, around the number from which the rows are found from the entries, in
    blocks with fewer and with more workgroups of entries than of rows to clear.  Whole numbers: the sums are exact in any order."""
    import compressgnn_runtime as rt
    rng = np.random.default_rng(width)
    blocks = [(gap + 2, {0: 3, gap + 1: 2}) for gap in (1790, 2045, 2046, 2047, 2048, 2049, 2304, 40000)]
    blocks += [(90000, {int(r): int(n) for r, n in zip(rng.choice(90000, 700, replace=False), rng.integers(1, 9, 700))}),
               (90000, {**{r: 5 for r in range(300)}, **{90000 - 1 - r: 70 for r in range(300)}}),
               (9000, {**{r: 1 for r in range(0, 9000, 5)}, 4500: 3000}), (70000, {1: 64, 35000: 65, 69998: 2000}),
               (600000 if width <= 33 else 60000, {0: 1})]
    for rows, taken in blocks:
        lens, v, e = rows_with_entries(rows, taken, rng)
        w = torch.from_numpy(rng.integers(-3, 4, len(e))).to(DEV).to(dtype)
        x = torch.from_numpy(rng.integers(-8, 9, (300, width))).to(DEV).to(dtype)
        at = torch.from_numpy(np.repeat(np.arange(rows), lens)).to(DEV)
        want = torch.zeros(rows, width, device=DEV, dtype=dtype).index_add_(0, at, x[e] * w[:, None])
        for _ in range(2):
            torch.full((rows, width), float("nan"), device=DEV, dtype=dtype)  # what the result may be given the memory of
            assert torch.equal(rt.spmm_func(v, e, w, x, "auto", None), want)
        base = torch.from_numpy(rng.integers(-9, 9, (rows, width))).to(DEV).to(dtype)
        assert torch.equal(rt.spmm_func(v, e, w, x, "auto", base.clone()), base + want)


@pytest.mark.parametrize("width", [1, 64])
def test_products_of_int64_arrays_are_not_held_up_by_empty_rows(width):
    """10^6 rows without entries: in the middle of 10^5 entries they cost what they cost behind them, and with few
    entries, whose workgroups are few, no more than with a million.  Four times as long is allowed; a workgroup that walks the rows
    between its entries, or few that clear all rows, take 20 times as long and more."""
    import compressgnn_runtime as rt
    rng = np.random.default_rng(1)
    rows, half = 1000003, 6250

    def time_of(taken):
        _, v, e = rows_with_entries(rows, taken, rng)
        w, x = torch.ones(len(e), device=DEV), torch.ones(300, width, device=DEV)
        times = []
        for _ in range(9):
            begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            begin.record()
            for _ in range(4):
                rt.spmm_func(v, e, w, x, "auto", None)
            end.record()
            end.synchronize()
            times.append(begin.elapsed_time(end))
        return sorted(times)[4]

    behind = time_of({r: 8 for r in range(2 * half)})
    between = time_of({**{r: 8 for r in range(half)}, **{rows - 1 - r: 8 for r in range(half)}})
    many, few = time_of({r: 1 for r in range(rows)}), time_of({r: 8 for r in range(125)})
    assert between < 4 * behind and few < 4 * many, (behind, between, many, few)


@pytest.mark.parametrize("rows,clusters,width,bias", [(6, 5, 100, False), (5, 9, 40, True), (3000, 70, 33, True), (3000, 70, 256, False),
                                                      (1 << 19, 1 << 14, 32, True), (1 << 18, 1 << 13, 100, False)])
def test_what_a_reconstruct_keeps_is_written(rows, clusters, width, bias):
    """Hooks on saved tensors are shown one bit per element in a tensor with a row of words per row of the output, and the same
    words each time, whatever the memory held before."""
    from CompressgnnReconstruct import Compressgnn_Reconstruct
    gen = torch.Generator(device=DEV).manual_seed(rows)
    used = clusters - clusters // 3  # the others have no rows
    ids = torch.randint(0, used, (rows,), device=DEV, generator=gen)
    reps = torch.randn(clusters, width, device=DEV, generator=gen, requires_grad=True)
    add = torch.randn(width, device=DEV, generator=gen, requires_grad=True) if bias else None
    grad = torch.randn(rows, width, device=DEV, generator=gen)
    inputs = (reps, add) if bias else (reps,)
    words, seen = (width + 31) // 32, []
    for left_over in (-1, 0x55555555):
        kept = []
        for n in (rows, clusters):  # what is kept may be given the memory of
            torch.full((n, words), left_over, device=DEV, dtype=torch.int32)
        with torch.autograd.graph.saved_tensors_hooks(lambda t: kept.append(t) or t, lambda t: t):
            out = Compressgnn_Reconstruct()(reps, ids, bias=add, activation="relu")
        assert sorted((tuple(t.shape), t.dtype) for t in kept) == sorted([((rows,), torch.int64), ((rows, words), torch.int32)])
        seen += [t for t in kept if t.dtype == torch.int32]
        got = torch.autograd.grad(out, inputs, grad)
    assert torch.equal(*seen)
    want = reps.index_select(0, ids)
    want = (want if add is None else want + add).relu()
    assert torch.equal(out, want)
    for a, b in zip(got, torch.autograd.grad(want, inputs, grad)):
        torch.testing.assert_close(a, b, atol=1e-5 * float(b.abs().max()), rtol=1e-4)  # sums of up to 2^19 numbers in another order


@pytest.mark.parametrize("rows,clusters,width,of_groups", [
    (1 << 19, 1 << 17, 32, True), (1 << 19, (1 << 17) + 1, 32, False), (1 << 19, 1 << 17, 31, True), (1 << 19, 1 << 15, 33, True),
    (1 << 19, (1 << 15) + 1, 33, False), (65536, 16384, 256, True), (65536, 16385, 256, False), (65536, 30000, 300, False),
    (20000, 20000, 64, False), (5000, 20000, 64, False), (3000, 3, 225, True)])
def test_which_bits_a_reconstruct_keeps(rows, clusters, width, of_groups):
    """Those of the representatives from 16 rows each on, 4 where a row is one word or whole ones, those of the rows otherwise:
    told by the memory that is held between the passes.  The gradient is that of the operator, bit for bit.  Without a
    gradient nothing is kept or made."""
    import compressgnn_runtime as rt
    from CompressgnnReconstruct import Compressgnn_Reconstruct
    gen = torch.Generator(device=DEV).manual_seed(rows)
    ids = torch.randint(0, clusters, (rows,), device=DEV, generator=gen)
    reps = torch.randn(clusters, width, device=DEV, generator=gen, requires_grad=True)
    grad = torch.randn(rows, width, device=DEV, generator=gen)
    out, signs = rt.cluster_reconstruct_signs(reps.detach(), ids, None, None)
    want = rt.cluster_reconstruct_backward_signs(grad, ids, signs, clusters, None)
    words = signs.size(1)

    def held(mode):
        Compressgnn_Reconstruct()(reps, ids, activation="relu")  # what is made once per index is there
        torch.cuda.synchronize()
        gc.collect()
        before = _requested()  # what tensors ask for: what they are given depends on the blocks that earlier tests left
        with mode:
            layer = Compressgnn_Reconstruct()(reps, ids, activation="relu")
        assert torch.equal(layer, out)
        return layer, _requested() - before - 4 * rows * width

    layer, kept = held(torch.enable_grad())
    assert kept == 4 * (clusters if of_groups else rows) * words
    assert torch.equal(torch.autograd.grad(layer, reps, grad)[0].view(torch.int32), want.view(torch.int32))
    del layer
    assert held(torch.no_grad())[1] == 0
