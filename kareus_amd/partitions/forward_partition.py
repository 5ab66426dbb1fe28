"""Forward execution of one partition.

Follows kareus/megatron/core/partitions/forward_partition.py:30-127: per op create
the context, gather inputs by port, decide ``requires_grad``, release the
hand-over when the scheduled op index is reached, run the op, record the release
event right after op ``start-1``, store outputs by port; afterwards run a
non-overlapped hand-over if ``start == -1`` and finally sync and publish its
result into the other nanobatch's store.
"""

from __future__ import annotations

from dataclasses import dataclass

from .context_manager import NanoBatchContext
from .op_context import operator_parameters
from .partition_base import PartitionBase


@dataclass
class ForwardPartition(PartitionBase):
    # adjacent ops that offer a fused forward (fc1 + the SwiGLU activation behind it) run as one
    # call; the numbers are those of the separate calls
    fuse_forward_ops: bool = True

    def _find_chains(self, plans):
        from ..operators.chains import forward_chains

        return forward_chains(plans, self.read_twice)

    def execute(self, ctx: NanoBatchContext, pre_ctx: NanoBatchContext) -> None:
        with self._on_stream(ctx), self._timed():
            self._execute(ctx, pre_ctx)

    def _execute(self, ctx: NanoBatchContext, pre_ctx: NanoBatchContext) -> None:
        start, _end, sm_num, block_size = self._setup_comm(ctx)
        store = ctx.tensor_store
        get, put, needs = store.get, store.set, store.needs_grad
        sinks = ctx.output_sinks
        timed = PartitionBase.timer is not None
        comm_out, comm_extra = None, []

        plans = self._plans()
        chains = self._op_chains if ctx.chains and not timed and self.fuse_forward_ops else None
        identity = self.comm_op is not None and len(self.comm_op.output_ports) == 1 and self._is_identity(pre_ctx)
        grad = self.is_grad_enabled
        idx, num_ops = 0, len(plans)
        while idx < num_ops:
            plan = plans[idx]
            x = get(plan.first_in)
            if start == idx and not identity:
                comm_out, comm_extra = self._launch_comm(pre_ctx, sm_num, block_size)
            chain = chains[idx] if chains is not None else None
            if (chain is not None and not idx < start < idx + chain.length and ctx.output_id not in chain.inside
                    and (not grad or needs(plan.first_in))
                    and chain.run(ctx, store, x, grad)):
                idx += chain.length
                if idx == start and not identity and not self._in_order(ctx):
                    self.comm_op.event_record(self._here())
                continue
            extras = [tuple([get(t) for t in plan.extra_ids])] if plan.extra_ids else []
            # the op behind this one runs in the same call when the two offer a fused forward and the
            # scheduled launch point does not fall between them
            group = [plan]
            if (plan.forward_pair and self.fuse_forward_ops and start != idx + 1
                    and plan.operator.can_fuse_forward_with(plans[idx + 1].operator)):
                group.append(plans[idx + 1])

            needs_grad = self.is_grad_enabled and (
                any([needs(t) for t in plan.in_ids])
                or any(p.requires_grad for member in group for p in operator_parameters(member.operator))
            )
            group_ctxs = []
            for member in group:
                op_ctx = ctx.create_op_context(member.op_id)
                op_ctx.requires_grad = needs_grad
                if ctx.in_line:
                    op_ctx.alone = True
                if sinks and member.op_id in sinks:
                    op_ctx.out_sink = sinks.pop(member.op_id)
                group_ctxs.append(op_ctx)
            k = len(group)
            last = idx + k - 1

            x, extra_out = plan.operator.fuser_forward(
                group_ctxs,
                x,
                basic_op_extra_inputs=extras if k == 1 else [extras[0] if extras else (), ()],
                basic_op_prev_ops=[None] * k,
                basic_op_next_ops=[None] * k,
                basic_op_kwargs=[{}] if k == 1 else [{}, {}],
            )

            if timed:
                for j in range(k):
                    self._op_done(idx + j)
            if last == start - 1 and not identity and not self._in_order(ctx):
                self.comm_op.event_record(self._here())

            tail = group[-1]
            put(tail.first_out, x, needs_grad)
            if tail.extra_out_ids and extra_out and extra_out[-1]:
                for tid, extra in zip(tail.extra_out_ids, extra_out[-1]):
                    if extra is not None:
                        put(tid, extra, needs_grad)
            idx = last + 1

        if identity:
            self._hand_on(pre_ctx, sm_num, block_size)
        elif self.comm_op is not None:
            if start == -1:
                comm_out, comm_extra = self._launch_comm_no_overlap(pre_ctx, sm_num, block_size)
            self._sync_comm(pre_ctx, comm_out, comm_extra)
