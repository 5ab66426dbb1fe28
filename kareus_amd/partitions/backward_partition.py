"""Backward execution of one partition.

Follows kareus/megatron/core/partitions/backward_partition.py:36-145: ops come from
the backward graph (already reversed, channels ``grad_*``); each looks up the
context its forward twin filled (same ``op_id``), stops the partition early when
that context needs no gradient, returns parameter gradients keyed by ``op_id`` and
frees the saved activations of every op as soon as it has run (kept in
``profiling_mode`` so one forward can feed many timed backward runs; tensors whose
object id is in ``protected_tensor_ids`` are shared between nanobatches and kept).
"""

from __future__ import annotations

from dataclasses import dataclass
from typing import Dict, List, Optional

from .context_manager import NanoBatchContext
from .op_context import clear_tensor_data
from .partition_base import PartitionBase


@dataclass
class BackwardPartition(PartitionBase):
    # adjacent ops that offer a fused backward (RMSNorm + the residual fork in front of it) run
    # as one call; the numbers are those of the separate calls
    fuse_backward_ops: bool = True

    def _find_chains(self, plans):
        from ..operators.chains import backward_chains

        return backward_chains(plans, self.read_twice)

    def execute(
        self,
        ctx: NanoBatchContext,
        pre_ctx: NanoBatchContext,
        protected_tensor_ids: Optional[set] = None,
    ) -> Dict[int, List]:
        with self._on_stream(ctx), self._timed():
            return self._execute(ctx, pre_ctx, protected_tensor_ids or set())

    def _fusable_follower(self, plans, idx: int, start: int, ctx: NanoBatchContext):
        """The op after ``idx`` when the two can run as one fused backward: the first op offers it
        (``can_fuse_backward_with``), the second consumes the first's only output and needs a
        gradient, and the scheduled launch point does not fall between them."""
        plan = plans[idx]
        if not plan.backward_pair or not self.fuse_backward_ops or start == idx + 1:
            return None
        nxt = plans[idx + 1]
        if not plan.operator.can_fuse_backward_with(nxt.operator):
            return None
        if not ctx.get_op_context(nxt.op_id).requires_grad:
            return None
        if any([t not in ctx.tensor_store for t in nxt.extra_ids]):
            return None
        return nxt

    def _execute(self, ctx, pre_ctx, protected: set) -> Dict[int, List]:
        start, _end, sm_num, block_size = self._setup_comm(ctx)
        store = ctx.tensor_store
        get, put = store.get, store.set
        timed = PartitionBase.timer is not None
        comm_out, comm_extra = None, []
        launched = False
        grad_params: Dict[int, List] = {}

        plans = self._plans()
        chains = self._op_chains if ctx.chains and not timed and self.fuse_backward_ops and not self.profiling_mode else None
        identity = self.comm_op is not None and len(self.comm_op.output_ports) == 1 and self._is_identity(pre_ctx)
        idx, num_ops = 0, len(plans)
        while idx < num_ops:
            op = plans[idx]
            op_ctx = ctx.get_op_context(op.op_id)
            if not op_ctx.requires_grad:
                break

            dy = get(op.first_in)
            if start == idx and not identity:
                comm_out, comm_extra = self._launch_comm(pre_ctx, sm_num, block_size, backward=True)
                launched = True
            chain = chains[idx] if chains is not None else None
            if chain is not None and not idx < start < idx + chain.length and ctx.output_id not in chain.inside:
                got = chain.run(ctx, store, dy, protected)
                if got is not None:
                    grad_params.update(got)
                    idx += chain.length
                    if idx == start and not identity and not self._in_order(ctx):
                        self.comm_op.event_record(self._here())
                    continue
            group, group_ctxs = [op], [op_ctx]
            grad_extra_out = [tuple([get(t) for t in op.extra_ids])] if op.extra_ids else []
            follower = self._fusable_follower(plans, idx, start, ctx)
            if follower is not None:
                group.append(follower)
                group_ctxs.append(ctx.get_op_context(follower.op_id))
                grad_extra_out = [tuple([get(t) for t in op.extra_ids]), tuple([get(t) for t in follower.extra_ids])]
            last = idx + len(group) - 1

            dx, op_param_grads, grad_extra_in = op.operator.fuser_backward(
                group_ctxs, dy, basic_op_grad_extra_outputs=grad_extra_out
            )

            for k, (member, member_ctx) in enumerate(zip(group, group_ctxs)):
                grad_params[member.op_id] = list(op_param_grads[k]) if len(group) > 1 else [
                    g for grads in op_param_grads for g in grads]
                if not self.profiling_mode:
                    if member_ctx.saved_tensors is not None:
                        clear_tensor_data(
                            *[t for t in member_ctx.saved_tensors if t is not None and id(t) not in protected]
                        )
                    member_ctx.saved_tensors = None
                if timed:
                    self._op_done(idx + k)
            if last == start - 1 and not identity and not self._in_order(ctx):
                self.comm_op.event_record(self._here())

            put(group[-1].first_out, dx)
            # gradients of extra inputs: every member of a fused group may have some (a projection
            # that adds the residual in its epilogue hands the residual's gradient on)
            for k, member in enumerate(group):
                extras_k = grad_extra_in[k] if (grad_extra_in and len(grad_extra_in) == len(group)) else (
                    grad_extra_in[-1] if (grad_extra_in and k == len(group) - 1) else ())
                for tid, g in zip(member.extra_out_ids, extras_k):
                    if g is not None:
                        put(tid, g)
            idx = last + 1

        if identity:
            self._hand_on(pre_ctx, sm_num, block_size)
        elif self.comm_op is not None:
            if not launched:  # no slot given, or the op loop stopped before reaching it
                comm_out, comm_extra = self._launch_comm_no_overlap(
                    pre_ctx, sm_num, block_size, backward=True
                )
            self._sync_comm(pre_ctx, comm_out, comm_extra)
        return grad_params
