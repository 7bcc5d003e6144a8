"""Multi-phase propagation over an edge-list (graph_type="coo") compressed graph.

The reference runs one gather + scatter-add per phase (layer/CompressgnnPropagation.py:68-83,
phases from loader/CompressgnnData.py:86-139): out[(V+R) x F] starts at zero, phase 0
gathers from x, phase k >= 1 from out, every phase adds weight * feature[src] into
out[dst]; the result is out[:V].

In the phases the loader makes, every edge that leaves a rule does so after the last one that reaches it.
The sum then is that of the compressed chain: the rules' values first (phase 0 into the rules, then
the edges from rule to rule in the order of their phases), then every vertex from its vertex and its rule
inputs at once.  Such a list becomes a PropagationPlan, whose kernels write every row once, with the
V x F result where the phases keep a (V+R) x F buffer (100,003 vertices, 64 features, forward and gradient:
118 us as one product per phase, 86 us so).

A phase list from elsewhere may have another shape.  Then every phase is one CSR product: its edges are grouped
by destination once (stable, so a destination sums its messages in edge order), and the gradient runs the
transposed phases in reverse order.  Where a source of phase k receives nothing in phase k the product of a
phase k >= 1 accumulates in place; a phase that breaks that too runs as a fresh product followed by an addition,
which is what the reference's gather-then-scatter computes for any phase list.
"""
import _paths  # noqa: F401
import numpy as np
import torch

import compressgnn_runtime as _native
from compress_graph import CompressGraph
from compressgnn_offline import csr_fold_levels, csr_fold_levels_bound, csr_transpose


def _grouped(keys, groups, others, weights):
    """The edges grouped by keys (stable, on the device): (row pointers, others, weights, positions)."""
    one_each = torch.arange(keys.numel() + 1, device=keys.device)
    rowptr, position, values = _native.csr_transpose(one_each, keys, weights, groups)
    return rowptr, others.index_select(0, position), values, position


def _levels(base, blocks):
    """(folded base, None) or (base, blocks): the rule levels multiplied into the rule stage where that stays
    within the bounds CompressGraph.plan() folds by.  Host CSR triples; blocks in the order they apply."""
    stored = len(base[1]) + sum(len(b[1]) for b in blocks)
    if (len(blocks) <= CompressGraph.max_fold_depth
            and csr_fold_levels_bound(base, blocks) <= CompressGraph.max_fold_growth * max(stored, 1)):
        return csr_fold_levels(base, blocks), None
    return base, blocks


class _Edges:
    """All phases as one edge list on the device, and whether it is a compressed chain."""

    def __init__(self, edge_index, edge_weight, V, R):
        self.V, self.R, self.phases = V, R, len(edge_index)
        device = edge_index[0].device  # where the others are taken to
        ends = torch.cat([e.detach().to(device) for e in edge_index], 1).to(torch.int64)
        self.src, self.dst = ends[0].contiguous(), ends[1].contiguous()
        counts = [e.size(1) for e in edge_index]
        self.weight = torch.cat([torch.ones(n, device=device) if edge_weight is None or edge_weight[k] is None
                                 else edge_weight[k].detach().to(device, torch.float32)
                                 for k, n in enumerate(counts)])
        self.phase = torch.repeat_interleave(torch.arange(self.phases, device=device),
                                             torch.tensor(counts, device=device), output_size=sum(counts))

    def is_chain(self):
        """(vertices are sources of phase 0 only and rules of the others, and every rule is complete before it is
        a source; whether there are edges from rule to rule).  One host read."""
        V, R, late = self.V, self.R, self.phase > 0
        if self.src.numel() == 0:
            return False, False
        from_rule, to_rule = self.src >= V, self.dst >= V
        in_range = ((self.src >= 0) & (self.dst >= 0) & (self.src < V + R) & (self.dst < V + R)).all()
        ruled = (late == from_rule).all()
        ordered = torch.ones((), dtype=torch.bool, device=self.src.device)
        if R > 0:
            leaving, reaching = torch.nonzero(from_rule).flatten(), torch.nonzero(to_rule).flatten()
            rule = lambda ids: (ids - V).clamp(0, R - 1)
            never, last = torch.full((R,), self.phases, device=self.src.device), torch.full((R,), -1, device=self.src.device)
            used = never.scatter_reduce(0, rule(self.src[leaving]), self.phase[leaving], 'amin')
            reached = last.scatter_reduce(0, rule(self.dst[reaching]), self.phase[reaching], 'amax')
            ordered = (reached < used).all()
        chain, levels = torch.stack([in_range & ruled & ordered, (from_rule & to_rule).any()]).tolist()
        return chain, levels

    def plan(self, levels, dtype=torch.float32):
        """The chain as a PropagationPlan for features of `dtype` (levels, as is_chain() reports)."""
        V, R, device = self.V, self.R, self.src.device
        forward = _grouped(self.dst, V + R, self.src, self.weight)
        # the gradient of a vertex: from its vertex targets first, then from its rule targets
        order = torch.cat([torch.nonzero(self.dst < V).flatten(), torch.nonzero(self.dst >= V).flatten()])
        src, dst, weight = (t.index_select(0, order) for t in (self.src, self.dst, self.weight))
        backward = _grouped(src, V + R, dst, weight)
        csr = lambda ptr, other, value, *rest: _native.DeviceCsr(ptr, other, value.to(dtype), *rest)
        cut = torch.stack([forward[0][V], backward[0][V]]).tolist()

        def vertex_rows(grouped, n):
            return csr(grouped[0][:V + 1].contiguous(), grouped[1][:n], grouped[2][:n], V, V + R, device, 32)

        def rule_rows(grouped, n, phase, seg, forwards):
            rowptr, other, value = grouped[0][V:] - n, grouped[1][n:], grouped[2][n:]
            if not levels:
                return csr(rowptr.contiguous(), other.contiguous(), value.contiguous(), R, V, device, seg), []
            rows = torch.repeat_interleave(torch.arange(R, device=device), rowptr[1:] - rowptr[:-1]).cpu().numpy()
            other, value, phase = (t.cpu().numpy() for t in (other, value, phase.index_select(0, grouped[3][n:])))
            level = np.where(other >= V, phase, 0)

            def part(k):
                keep = level == k
                ptr = np.concatenate([[0], np.cumsum(np.bincount(rows[keep], minlength=R))])
                return ptr, other[keep] - (V if k else 0), value[keep]

            blocks = [part(k) for k in range(1, self.phases)]
            base, blocks = _levels(part(0), blocks if forwards else blocks[::-1])
            t = torch.from_numpy
            if blocks is not None and not forwards:
                blocks = blocks[::-1]  # a plan runs the levels of the gradient from the last to the first
            return (csr(t(base[0]), t(base[1]), t(base[2]), R, V, device, seg),
                    [csr(t(b[0]), t(b[1]), t(b[2]), R, R, device, 32) for b in blocks or []])

        rules, up = rule_rows(forward, cut[0], self.phase, 16, True)
        rules_back, down = rule_rows(backward, cut[1], self.phase.index_select(0, order), 32, False)
        if len(up) != len(down):  # folded one way only: the levels of the other way as empty products
            return None
        plan = _native.PropagationPlan(V, R, rules, up, rules_back, down)
        plan.set_vertex_stages(vertex_rows(forward, cut[0]), vertex_rows(backward, cut[1]))
        return plan


class CooPhasePlan:
    """The chain of a phase list, or device CSR blocks of its phases: by destination (forward) and by source
    (gradient)."""

    def __init__(self, edge_index, edge_weight, vertex_cnt, rule_cnt):
        if len(edge_index) == 0:
            raise ValueError("expected at least one phase")
        if edge_weight is not None and len(edge_weight) != len(edge_index):
            raise ValueError("edge_weight must hold one tensor per phase")
        self.V, self.R = int(vertex_cnt), int(rule_cnt)
        total = self.V + self.R
        device = edge_index[0].device
        if device.type != "cuda":
            raise RuntimeError("multi-phase propagation runs on the GPU only: move the data to a GPU")
        self.device = device
        self.forward_blocks, self.backward_blocks = [], []
        self.in_place = []  # per phase: no node is both a source and a destination of the phase
        # keeps the tensors (and so their addresses) alive for as long as the plan is cached
        self.sources = (list(edge_index), None if edge_weight is None else list(edge_weight))
        for k, edges in enumerate(edge_index):
            if edges.dim() != 2 or edges.size(0) != 2:
                raise ValueError("every phase must be a [2, E] edge tensor")
            if edge_weight is not None and edge_weight[k] is not None and edge_weight[k].shape != edges[0].shape:
                raise ValueError("edge_weight[%d] must have one value per edge" % k)
        edges = _Edges(edge_index, edge_weight, self.V, self.R)
        is_chain, self._levels = edges.is_chain()
        self.chain = edges.plan(self._levels) if is_chain else None
        # weights are of 32 bits; without any the sums take features of either precision
        self._wide_chain, self._weighted = None, edge_weight is not None and any(w is not None for w in edge_weight)
        if self.chain is not None:
            return
        t = torch.from_numpy
        for k, edges in enumerate(edge_index):
            src = edges[0].detach().cpu().numpy().astype(np.int64)
            dst = edges[1].detach().cpu().numpy().astype(np.int64)
            w = None
            if edge_weight is not None and edge_weight[k] is not None:
                w = edge_weight[k].detach().cpu().numpy().astype(np.float32)
            cols = self.V if k == 0 else total  # phase 0 gathers from x
            rows_back = cols
            if src.size and (src.min() < 0 or src.max() >= cols or dst.min() < 0 or dst.max() >= total):
                raise ValueError("phase %d: node id out of range" % k)
            is_src = np.zeros(total, bool)
            is_src[src] = True
            self.in_place.append(not bool(is_src[dst].any()))
            # by source (stable): the transposed block used by the gradient
            by_src = np.argsort(src, kind="stable")
            sp = np.zeros(rows_back + 1, np.int64)
            np.cumsum(np.bincount(src, minlength=rows_back), out=sp[1:])
            s_col, s_val = dst[by_src], None if w is None else w[by_src]
            # by destination, ties in edge order: the forward block
            dp, d_col, d_val = csr_transpose(sp, s_col, s_val, total)
            wt = lambda a: None if a is None else t(np.ascontiguousarray(a))
            self.forward_blocks.append(_native.DeviceCsr(t(dp), t(d_col), wt(d_val), total, cols, device))
            self.backward_blocks.append(_native.DeviceCsr(t(sp), t(np.ascontiguousarray(s_col)), wt(s_val),
                                                          rows_back, total, device))

    def chain_for(self, dtype):
        """The chain for features of this type: an unweighted list holds a one of the type for every edge."""
        if dtype != torch.float64 or self._weighted:
            return self.chain
        if self._wide_chain is None:
            self._wide_chain = _Edges(self.sources[0], None, self.V, self.R).plan(self._levels, dtype)
        return self._wide_chain

    def forward(self, x):
        x = x.contiguous()
        if x.dim() != 2 or x.size(0) != self.V:
            raise ValueError("x must be [vertex_cnt, F]")
        if self.chain is not None:
            return self.chain_for(x.dtype).forward(x)
        out = self.forward_blocks[0].spmm(x)
        for block, in_place in zip(self.forward_blocks[1:], self.in_place[1:]):
            out = block.spmm(out, out) if in_place else out + block.spmm(out)
        return out[:self.V]

    def backward(self, grad):
        grad = grad.contiguous()
        if self.chain is not None:
            return self.chain_for(grad.dtype).backward(grad)
        if len(self.backward_blocks) == 1:
            full = grad if self.R == 0 else torch.cat([grad, grad.new_zeros((self.R, grad.size(1)))])
            return self.backward_blocks[0].spmm(full)
        full = torch.cat([grad, grad.new_zeros((self.R, grad.size(1)))])
        for block, in_place in zip(reversed(self.backward_blocks[1:]), reversed(self.in_place[1:])):
            full = block.spmm(full, full) if in_place else full + block.spmm(full)
        return self.backward_blocks[0].spmm(full)


class CooPropagateFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, plan, x):
        ctx.plan = plan
        return plan.forward(x)

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, grad):
        return None, ctx.plan.backward(grad)


def coo_propagate(plan, x):
    """plan.forward(x) with its gradient; a chain's step of autograd is native."""
    if plan.chain is None or x.dim() != 2 or x.size(0) != plan.V:
        return CooPropagateFunction.apply(plan, x)
    out = _native.propagate(plan.chain_for(x.dtype), x, once_differentiable=True)
    return CooPropagateFunction.apply(plan, x) if out is None else out


class CooPlanCache:
    """Plans keyed by the identity of the phase tensors (addresses, versions, shapes)."""

    def __init__(self, limit=4):
        self.limit = limit
        self.entries = {}

    @staticmethod
    def _key(edge_index, edge_weight, vertex_cnt, rule_cnt):
        sig = lambda t: None if t is None else (t.data_ptr(), t._version, tuple(t.shape), str(t.device))
        weights = () if edge_weight is None else tuple(sig(w) for w in edge_weight)
        return (tuple(sig(e) for e in edge_index), weights, int(vertex_cnt), int(rule_cnt))

    def get(self, edge_index, edge_weight, vertex_cnt, rule_cnt):
        key = self._key(edge_index, edge_weight, vertex_cnt, rule_cnt)
        plan = self.entries.get(key)
        if plan is None:
            if len(self.entries) >= self.limit:
                self.entries.pop(next(iter(self.entries)))
            plan = self.entries[key] = CooPhasePlan(edge_index, edge_weight, vertex_cnt, rule_cnt)
        return plan
