"""The operators between two schedule points, run as one native call.

A partition holds the same few operator sequences over and over: residual fork, norm, QKV projection, QKV split, rotary
embedding, attention, out-projection; residual fork, norm, fc1, activation, fc2; and the same projections backward.  The
engine finds them when it looks a partition's graph up, and, where nothing asks for the steps in between, has the native host
side run the launches of the whole sequence.  The launches, their order, their plans and their results are those of the
operators one by one, every operator's context holds what the operator itself would have saved (a pass may run forward one
way and backward the other), and saved activations are dropped at the same points.  One operator at a time the interpreter
spent 6-10 us per operator around launches of 3-5 us.

A sequence runs operator by operator whenever something looks inside it or is not the stock case: another reader of a tensor
between its operators, a timer or a schedule's launch point there, an operator, its class, an operator method or a backend
method that was replaced, another backend, frozen weights, operands that the kernels do not address in place, a trace.  (Reference for what the operators do:
kareus/megatron/core/transformer/transformer_layer.py:148-174 and the files each operator names.)
"""

from __future__ import annotations

import math
from typing import List, Optional, Tuple

import torch

from ..backend import get_backend, reserved_compute_units
from ..partitions.op_context import clear_tensor_data
from .attention import TEDotProductAttentionOp
from .bias_dropout_add import BiasDropoutAddOp
from .bias_swiglu import BiasSwigluOp
from .linear import PartitionableLinear, TEColumnParallelLinearOp, TERowParallelLinearOp
from .qkv_postprocess import QKVPostProcessOp
from .residual_fork import ResidualForkOp
from .rmsnorm import PartitionableRMSNorm
from .rotary_embedding import RotaryEmbeddingOp

_FORWARD_ATTENTION = (ResidualForkOp, PartitionableRMSNorm, TEColumnParallelLinearOp, QKVPostProcessOp, RotaryEmbeddingOp,
                      TEDotProductAttentionOp, TERowParallelLinearOp)
_FORWARD_MLP = (ResidualForkOp, PartitionableRMSNorm, TEColumnParallelLinearOp, BiasSwigluOp, TERowParallelLinearOp)
_BACKWARD_MLP = (TERowParallelLinearOp, BiasSwigluOp, TEColumnParallelLinearOp)
_BACKWARD_ATTENTION = (TERowParallelLinearOp, TEDotProductAttentionOp, RotaryEmbeddingOp, QKVPostProcessOp, TEColumnParallelLinearOp)

#: what the operators of a chain call, as this package defines it: anything else runs operator by operator
_METHODS = {
    ResidualForkOp: frozenset(("fuser_forward",)),
    PartitionableRMSNorm: frozenset(("fuser_forward", "op_forward")),
    TEColumnParallelLinearOp: frozenset(("fuser_forward", "op_forward", "fuser_backward", "op_backward", "_split", "_weight_grad",
                                         "can_fuse_forward_with")),
    TERowParallelLinearOp: frozenset(("fuser_forward", "op_forward", "fuser_backward", "op_backward", "_split", "_weight_grad",
                                      "can_fuse_backward_with")),
    QKVPostProcessOp: frozenset(("fuser_forward", "fuser_backward", "split", "merge")),
    RotaryEmbeddingOp: frozenset(("fuser_forward", "fuser_backward", "_shared_fused")),
    TEDotProductAttentionOp: frozenset(("fuser_forward", "fuser_backward")),
    BiasSwigluOp: frozenset(("fuser_forward", "op_forward", "fuser_backward", "op_backward")),
    BiasDropoutAddOp: frozenset(("fuser_forward", "fuser_backward")),
}
_STOCK = tuple((cls, n, getattr(cls, n)) for cls, names in _METHODS.items() for n in sorted(names))
_BACKEND_METHODS = ("gemm", "linear_fwd", "linear_dgrad", "linear_wgrad", "linear_wgrad_segments", "wgrad_segments_ok",
                    "MAX_WGRAD_SEGMENTS", "rows_view", "rows_in_place", "_operand", "rmsnorm_fwd",
                    "split_qkv", "qk_norm_fwd", "qk_norm_bwd", "rope_fused_inplace", "attn_fwd", "attn_bwd", "swiglu_fwd",
                    "can_fuse_swiglu", "can_fuse_swiglu_bwd", "MAX_RUN_ROWS", "_split_code", "_num_cus")
_BACKEND_STOCK: Tuple = ()   # (filled by the first pass, whole: other threads' first passes may be at it too)


def chains_allowed() -> bool:
    """Whether the operators' and the hip backend's methods are the package's own and nothing traces: asked once per pass."""
    global _BACKEND_STOCK
    if torch._C._get_tracing_state() is not None:
        return False
    for cls, name, fn in _STOCK:
        if getattr(cls, name) is not fn:
            return False
    be = get_backend("hip")
    cls = type(be)
    if not _BACKEND_STOCK:
        from ..backend import hip

        _BACKEND_STOCK = (*[(n, hip.STOCK[n]) for n in _BACKEND_METHODS], ("_n", hip.load_native()))
    own = be.__dict__
    for name, fn in _BACKEND_STOCK:
        if name in own:
            if name != "_n" or own[name] is not fn:
                return False
        elif cls.__dict__.get(name) is not fn:
            return False
    return True


def _matches(plans, at: int, classes) -> bool:
    if at + len(classes) > len(plans):
        return False
    before = None
    for p, c in zip(plans[at:at + len(classes)], classes):
        if type(p.operator) is not c or (before is not None and (before.first_out is None or before.first_out != p.first_in)):
            return False
        before = p
    return True


def _untouched(ops) -> bool:
    """No method of these operators was replaced on the instance, nor its class since the plans were made (parametrizations do
    that), and they run on the hip backend."""
    for op in ops:
        d = op.__dict__
        methods = _METHODS.get(type(op))
        if methods is None or d.get("_backend_name") != "hip" or not methods.isdisjoint(d):
            return False
    return True


def _max_cus(be, device) -> int:
    reserved = reserved_compute_units()
    return max(be._num_cus(device) - reserved, 8) if reserved else 0


def _split(be, linear, ctx_alone: bool) -> int:
    split_k = linear.split_k
    return be._split_code(True if (split_k is False and ctx_alone) else split_k)


class _Chain:
    """``inside``: the tensors between the operators, which are not put in the store."""

    def __init__(self, plans) -> None:
        self.plans = list(plans)
        self.length = len(self.plans)
        self.ops = [p.operator for p in self.plans]
        inside = self.inside = set()
        for p in plans:
            inside.update(p.out_ids)
        inside.difference_update(plans[0].extra_out_ids)
        inside.discard(plans[-1].first_out)


class _ForwardChain(_Chain):
    """``run`` returns whether the chain ran; the contexts are then filled and the outputs are in the store."""

    def _contexts(self, ctx, grad: bool) -> List:
        made = []
        for p in self.plans:
            c = ctx.create_op_context(p.op_id)
            c.requires_grad = grad
            if ctx.in_line:
                c.alone = True
            made.append(c)
        return made

    def _finish(self, ctx, store, x, y, sink, added: bool, grad: bool) -> None:
        first, last = self.plans[0], self.plans[-1]
        if sink is not None:
            del ctx.output_sinks[last.op_id]
            y = sink
        if added:
            y._kr_residual_added = True
        # (what the fork hands on beside the chain; the tensors between its operators are nobody else's: see _chains)
        for tid in first.extra_out_ids:
            store.set(tid, x, grad)
        store.set(last.first_out, y, grad)


class _ForwardBehindAdd:
    """The residual add in front of a chain, where the projection before it has added the residual already: it hands its
    input on."""

    def __init__(self, add, chain) -> None:
        self.plan, self.chain = add, chain
        self.length = chain.length + 1
        self.inside = chain.inside | {add.first_out}

    def run(self, ctx, store, x, grad: bool) -> bool:
        op = self.plan.operator
        if (not getattr(x, "_kr_residual_added", False) or (op.training and op.dropout_prob != 0.0) or not _untouched((op,))
                or (ctx.output_sinks and self.plan.op_id in ctx.output_sinks) or not self.chain.run(ctx, store, x, grad)):
            return False
        c = ctx.create_op_context(self.plan.op_id)
        c.requires_grad = grad
        if ctx.in_line:
            c.alone = True
        c.scale, c.has_bias = 1.0, False
        return True


class _ForwardAttention(_ForwardChain):
    def run(self, ctx, store, x, grad: bool) -> bool:
        fork, norm, qkv, post, rope, attn, proj = self.ops
        freqs = store.get(self.plans[4].extra_ids[1])
        if freqs is None or not isinstance(freqs, torch.Tensor) or not post.grouped_query_view or not _untouched(self.ops):
            return False
        be = get_backend("hip")
        sink = ctx.output_sinks.get(self.plans[6].op_id) if ctx.output_sinks else None
        added = proj.fuse_residual
        if sink is not None and not added:
            return False
        gq = gk = qn = post.q_layernorm
        if qn is not None:
            gq, gk = qn.weight, post.k_layernorm.weight
        hd = post.hd
        scale = attn.softmax_scale if attn.softmax_scale is not None else 1.0 / math.sqrt(hd)
        alone = ctx.in_line
        done = be._n.attn_chain_fwd(x, norm.weight, norm.eps, qkv.weight, gq, gk, float(qn.eps) if qn is not None else 0.0, freqs,
                                    post.ng, post.nq // post.ng, hd, scale, attn.beside_other_streams,
                                    _split(be, qkv, alone), proj.weight, _split(be, proj, alone), x if added else None, sink,
                                    _max_cus(be, x.device))
        if done is None:
            return False
        y, x2d, rstd, normed, q, k, v, o, lse, o2d, mixed, qk_rstd = done
        _, cn, cq, cp, cr, ca, co = self._contexts(ctx, grad)
        if grad:
            cn.to_save = (x2d, rstd)
            cq.to_save = (normed,)
            if mixed is not None:
                cp.to_save = (mixed, qk_rstd)
            cr.to_save = (freqs,)
            ca.to_save = (q, k, v, o, lse)
            ca.scale = scale
            co.to_save = (o2d,)
            cq.input_requires_grad = co.input_requires_grad = True
        self._finish(ctx, store, x, y, sink, added, grad)
        return True


class _ForwardMlp(_ForwardChain):
    def run(self, ctx, store, x, grad: bool) -> bool:
        fork, norm, fc1, act, fc2 = self.ops
        if not _untouched(self.ops):
            return False
        be = get_backend("hip")
        sink = ctx.output_sinks.get(self.plans[4].op_id) if ctx.output_sinks else None
        added = fc2.fuse_residual
        if sink is not None and not added:
            return False
        w1 = fc1.weight
        alone = ctx.in_line
        done = be._n.mlp_chain_fwd(x, norm.weight, norm.eps, w1, _split(be, fc1, alone),
                                   fc1.fuse_activation and be.can_fuse_swiglu(w1.shape[0]), fc2.weight, _split(be, fc2, alone),
                                   x if added else None, sink, _max_cus(be, x.device))
        if done is None:
            return False
        y, x2d, rstd, normed, pre, activated = done
        _, cn, c1, ca, c2 = self._contexts(ctx, grad)
        if grad:
            cn.to_save = (x2d, rstd)
            c1.to_save = (normed,)
            ca.to_save = (pre,)
            ca.ori_shape = (x.shape[0], x.shape[1], pre.shape[1])
            c2.to_save = (activated,)
            c1.input_requires_grad = c2.input_requires_grad = True
        self._finish(ctx, store, x, y, sink, added, grad)
        return True


class _BackwardChain(_Chain):
    """``run`` returns the parameter gradients by op id, or None where the chain did not run."""

    def _contexts(self, ctx) -> Optional[List]:
        """The operators' contexts, if every one needs a gradient."""
        ctxs = [ctx.op_contexts[p.op_id] for p in self.plans]
        for c in ctxs:
            if not c.requires_grad:
                return None
        return ctxs

    def _finish(self, store, ctxs, dy, dx, protected, released: bool) -> None:
        first, last = self.plans[0], self.plans[-1]
        if self.ops[0].fuse_residual:   # the residual input passes the incoming gradient through
            for tid in first.extra_out_ids:
                store.set(tid, dy)
        store.set(last.first_out, dx)
        left = []
        for c in ctxs:
            if not released and c.saved_tensors is not None:
                left.extend([t for t in c.saved_tensors if t is not None and id(t) not in protected])
            c.saved_tensors = None
        if left:
            get_backend("hip")._n.release(left)   # (op_context.clear_tensor_data)


class _BackwardBehindAdd:
    """A residual add without dropout in front of a chain: both its gradients are the incoming one."""

    def __init__(self, add, chain) -> None:
        self.plan, self.chain = add, chain
        self.length = chain.length + 1
        self.inside = chain.inside | {add.first_out}

    def run(self, ctx, store, dy, protected):
        c = ctx.op_contexts[self.plan.op_id]
        if not c.requires_grad or c.scale != 1.0 or not _untouched((self.plan.operator,)):
            return None
        got = self.chain.run(ctx, store, dy, protected)
        if got is None:
            return None
        for tid in self.plan.extra_out_ids:
            store.set(tid, dy)
        c.saved_tensors = None
        got[self.plan.op_id] = []
        return got


class _BetweenProjections:
    """A chain's first projection leaves the operands of its weight gradient over nanobatches on streams where the operators would:
    behind its own input gradient, so that the event is there, and the launch over all nanobatches, before the chain's others are
    enqueued.  (Behind the whole chain, two nanobatches of 4 x 4096 tokens of a 3/1-head shard took 1.3 % longer.)"""

    __slots__ = ("be", "linear", "ctx", "dy", "x", "dw")

    def __init__(self, be, linear, ctx, dy, x) -> None:
        self.be, self.linear, self.ctx, self.dy, self.x, self.dw = be, linear, ctx, dy, x, None

    def __call__(self) -> None:
        self.dw = PartitionableLinear._weight_grad(self.be, self.ctx, self.be.rows_in_place(self.dy), self.x,
                                                   self.linear._split(self.ctx))


def _between(be, linear, ctx, dy, x) -> Optional[_BetweenProjections]:
    sink = getattr(ctx, "wgrad_sink", None)
    return None if sink is None or sink.get("in_line") else _BetweenProjections(be, linear, ctx, dy, x)


def _add_pair(be, linear, ctx, dy, x):
    """The weight gradient of a projection over nanobatches.  On streams of their own it is PartitionableLinear._weight_grad.  On
    one stream the pair is left in the layer's sink without events, and the last nanobatch contracts all of them in nanobatch order."""
    sink = ctx.wgrad_sink
    n = sink["n"]
    if not sink.get("in_line") or not sink["defer"]:
        return PartitionableLinear._weight_grad(be, ctx, dy, x, linear._split(ctx))
    pairs = sink.get("pairs")
    if pairs is None:
        pairs = sink["pairs"] = []
    # (aliases: the storage behind the saved tensor objects is dropped; the record is the one that _weight_grad leaves without
    # events: another nanobatch of the pass may get here operator by operator)
    pairs.append((ctx.nanobatch_index, dy.detach(), x.detach(), None, None))
    if len(pairs) < n:
        return None
    pairs.sort(key=lambda p: p[0])
    sink["pairs"] = None
    sink["turn"][0] += 1
    dys, xs = [p[1] for p in pairs], [p[2] for p in pairs]
    dw = be._n.wgrad_segments(dys, xs, None, False, be._split_code(PartitionableLinear.wgrad_over_all_split_k),
                              _max_cus(be, dy.device))
    if dw is None:
        split_k = linear._split(ctx)
        dw = be.linear_wgrad(dys[0], xs[0], split_k=split_k)
        for d, v in zip(dys[1:], xs[1:]):
            be.linear_wgrad(d, v, out=dw, accumulate=True, split_k=split_k)
    return dw


class _BackwardMlp(_BackwardChain):
    def run(self, ctx, store, dy, protected):
        fc2, act, fc1 = self.ops
        ctxs = self._contexts(ctx)
        if ctxs is None or not fc2.fuse_activation or not _untouched(self.ops):
            return None
        c2, ca, c1 = ctxs
        w2, w1 = fc2.weight, fc1.weight
        if not (w2.requires_grad and w1.requires_grad):
            return None
        (activated,), (pre,), (normed,) = c2.saved_tensors, ca.saved_tensors, c1.saved_tensors
        be = get_backend("hip")
        alone = c2.alone
        here = getattr(c2, "wgrad_sink", None) is None
        between = _between(be, fc2, c2, dy, activated)
        done = be._n.mlp_chain_bwd(dy, w2, pre, activated, w1, normed, _split(be, fc2, alone), _split(be, fc1, alone), here,
                                   _max_cus(be, dy.device), between)
        if done is None:
            return None
        dx, dpre, dw2, dw1 = done
        if not here:
            dw2 = between.dw if between is not None else _add_pair(be, fc2, c2, be.rows_in_place(dy), activated)
            dw1 = _add_pair(be, fc1, c1, dpre, normed)
        self._finish(store, ctxs, dy, dx.view(*dy.shape[:-1], dx.shape[1]), protected, here)
        p2, pa, p1 = self.plans
        return {p2.op_id: [dw2], pa.op_id: [], p1.op_id: [dw1]}


class _BackwardAttention(_BackwardChain):
    def run(self, ctx, store, dy, protected):
        proj, attn, rope, post, qkv = self.ops
        ctxs = self._contexts(ctx)
        if ctxs is None or not _untouched(self.ops):
            return None
        co, ca, cr, cp, cq = ctxs
        wo, wq = proj.weight, qkv.weight
        if not (wo.requires_grad and wq.requires_grad):
            return None
        gq = gk = mixed = qk_rstd = None
        if post.q_layernorm is not None:
            gq, gk = post.q_layernorm.weight, post.k_layernorm.weight
            mixed, qk_rstd = cp.saved_tensors
        (o2d,), (q, k, v, o, lse), (freqs,), (normed,) = (co.saved_tensors, ca.saved_tensors, cr.saved_tensors, cq.saved_tensors)
        be = get_backend("hip")
        alone = co.alone
        here = getattr(co, "wgrad_sink", None) is None
        between = _between(be, proj, co, dy, o2d)
        done = be._n.attn_chain_bwd(dy, wo, q, k, v, o, lse, o2d, freqs, ca.scale, attn.beside_other_streams, mixed, qk_rstd,
                                    gq, gk, wq, normed, _split(be, proj, alone), _split(be, qkv, alone), here,
                                    _max_cus(be, dy.device), between)
        if done is None:
            return None
        dx, dmixed, dwo, dwq, dgq, dgk = done
        if not here:
            dwo = between.dw if between is not None else _add_pair(be, proj, co, be.rows_in_place(dy), o2d)
            dwq = _add_pair(be, qkv, cq, dmixed, normed)
        elif id(freqs) not in protected:
            clear_tensor_data(freqs)
        self._finish(store, ctxs, dy, dx.view(*dy.shape[:-1], dx.shape[1]), protected, here)
        po, pa, pr, pp, pq = self.plans
        return {po.op_id: [dwo], pa.op_id: [], pr.op_id: [], pp.op_id: [] if gq is None else [dgq, dgk], pq.op_id: [dwq]}


def _chains(plans, read_twice, find, behind_add) -> List:
    """By index, the chain that starts there, if one does: a chain, or a residual add and the chain behind it.  A chain reads each
    tensor between its operators once, so one that the graph reads twice (``read_twice``), or this partition, should one of its
    operators have been replaced by one with other ports, has another reader: no chain.  (Part of a new model's first pass: 100 us
    for a layer with two nanobatches.)"""
    if read_twice is None:
        return [None] * len(plans)
    found = [find(plans, at) for at in range(len(plans))]
    ids = [t for p in plans for t in p.in_ids]
    if len(set(ids)) != len(ids):
        read_twice = read_twice.union([t for t in ids if ids.count(t) > 1])
    for at, chain in enumerate(found):
        if chain is None:
            continue
        if not chain.inside.isdisjoint(read_twice):
            found[at] = None
        elif (at and type(plans[at - 1].operator) is BiasDropoutAddOp and plans[at - 1].first_out == plans[at].first_in
              and plans[at].first_in not in read_twice):
            found[at - 1] = behind_add(plans[at - 1], chain)
    return found


def forward_chains(plans, read_twice) -> List:
    """The chains of operators of a forward partition."""
    return _chains(plans, read_twice, _forward_chain, _ForwardBehindAdd)


def backward_chains(plans, read_twice) -> List:
    """The same for a backward partition."""
    return _chains(plans, read_twice, _backward_chain, _BackwardBehindAdd)


def _forward_chain(plans, at: int) -> Optional[_ForwardChain]:
    if _matches(plans, at, _FORWARD_ATTENTION):
        fork, norm, qkv, post, rope, attn, proj = plans[at:at + 7]
        if (len(rope.extra_ids) == 2 and rope.extra_ids[0] == post.extra_out_ids[0]
                and attn.extra_ids == (rope.extra_out_ids[0], post.extra_out_ids[1])
                and not norm.extra_ids and not qkv.extra_ids and proj.extra_ids in ((), fork.extra_out_ids[:1])
                and bool(proj.extra_ids) == bool(proj.operator.fuse_residual)):
            return _ForwardAttention(plans[at:at + 7])
    if _matches(plans, at, _FORWARD_MLP):
        fork, norm, fc1, act, fc2 = plans[at:at + 5]
        if (not norm.extra_ids and not fc1.extra_ids and fc2.extra_ids in ((), fork.extra_out_ids[:1])
                and bool(fc2.extra_ids) == bool(fc2.operator.fuse_residual)):
            return _ForwardMlp(plans[at:at + 5])
    return None


def _backward_chain(plans, at: int) -> Optional[_BackwardChain]:
    if _matches(plans, at, _BACKWARD_MLP):
        return _BackwardMlp(plans[at:at + 3])
    if _matches(plans, at, _BACKWARD_ATTENTION):
        proj, attn, rope, post, qkv = plans[at:at + 5]
        if (rope.extra_ids == attn.extra_out_ids[:1] and len(attn.extra_out_ids) == 2
                and post.extra_ids == (rope.extra_out_ids[0], attn.extra_out_ids[1])):
            return _BackwardAttention(plans[at:at + 5])
    return None
