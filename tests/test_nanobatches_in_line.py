"""Small nanobatches run one after the other on the caller's stream (``LayerConfig.nanobatches_in_line``)."""

import dataclasses
import os

import pytest
import torch

from kareus_amd import LayerConfig, LayerStack
from kareus_amd.operators.noop_collective import NoOpAllReduce
from kareus_amd.partitions import partition_base
from kareus_amd.partitions.streams import use_stream_api
from kareus_amd.scheduler import PipelineCommScheduler

gpu = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a HIP device")]


def _cfg(**kw):
    base = dict(hidden_size=4096, num_attention_heads=8, num_query_groups=2, kv_channels=128, ffn_hidden_size=3584)
    return LayerConfig(**{**base, **kw})


def test_the_rule_follows_the_size_of_a_nanobatch():
    own = _cfg(streams_are_own=True)
    assert own.nanobatches_in_line(256, 1) and own.nanobatches_in_line(1024, 1) and own.nanobatches_in_line(512, 2)
    assert not own.nanobatches_in_line(4096, 1) and not own.nanobatches_in_line(1024, 4)
    assert not _cfg().nanobatches_in_line(256, 1)                                    # a caller's own streams are used
    assert not _cfg(streams_are_own=True, backend="eager").nanobatches_in_line(256, 1)


class _NoDevice:
    """A stream interface whose streams are mere objects: enough to build a stack."""

    new_stream = new_event = current_stream = staticmethod(object)

    @staticmethod
    def available():
        return True


def _built(**kw):
    cfg = _cfg(hidden_size=64, num_attention_heads=2, num_query_groups=1, kv_channels=32, ffn_hidden_size=96, **kw)
    with use_stream_api(_NoDevice()):
        LayerStack(cfg)
    return cfg


def test_streams_that_a_caller_names_are_used_whenever_it_names_them():
    cfg = _built()
    assert len(cfg.nanobatch_streams) == 2 and cfg.nanobatches_in_line(256, 1)          # the driver's own
    assert dataclasses.replace(cfg).nanobatches_in_line(256, 1)
    assert not dataclasses.replace(cfg, nanobatch_streams=[object(), object()]).nanobatches_in_line(256, 1)
    cfg.nanobatch_streams[1] = object()                                                   # one of them
    assert not cfg.nanobatches_in_line(256, 1)
    cfg = _built()
    cfg.nanobatch_streams = [object(), object()]                                          # all, after the stack was built
    assert not cfg.nanobatches_in_line(256, 1)
    assert not _built(nanobatch_streams=[object(), object()]).nanobatches_in_line(256, 1)  # before


def test_a_plan_and_the_switch_keep_the_streams():
    """Under a plan the overlap windows order the streams and the resource shapes leave compute units to them."""
    cfg = _cfg(streams_are_own=True)
    assert cfg.nanobatches_in_line(256, 1)
    cfg.kareus_scheduler = object()
    assert not cfg.nanobatches_in_line(256, 1)
    assert not _cfg(streams_are_own=True, in_line_below_ms=0.0).nanobatches_in_line(8, 1)


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a HIP device")
def test_a_plan_reserves_compute_units_on_a_small_pass(fixtures_dir, monkeypatch):
    """The resource shapes of the shipped plan reach the partitions of a small layer: budgets are entered, as many
    as without the in-line rule, and the hand-overs record and wait."""
    budgets, waits = [], []
    reserve = partition_base.reserve_compute_units
    monkeypatch.setattr(partition_base, "reserve_compute_units", lambda n: budgets.append(n) or reserve(n))
    wait = NoOpAllReduce.event_wait
    monkeypatch.setattr(NoOpAllReduce, "event_wait", lambda self: waits.append(self.batch_idx) or wait(self))
    cfg = _cfg(hidden_size=1024, num_attention_heads=8, ffn_hidden_size=896, num_layers=2)
    model = LayerStack(cfg, device="cuda", seed=3)
    sch = PipelineCommScheduler(os.path.join(fixtures_dir, "scheds_pipeline_02328.py"), pp_rank=0, num_microbatches=8,
                                use_activation_checkpointing=True)
    cfg.kareus_scheduler = sch
    sch.on_step_begin()
    sch.on_instruction_begin("forward")
    model(torch.randn(256, 4, 1024, device="cuda", dtype=torch.bfloat16))
    torch.cuda.synchronize()
    assert budgets and waits


@pytest.mark.parametrize("nnb,b,s", [(2, 2, 256), (4, 4, 136), (2, 6, 200), (4, 8, 64)])
@pytest.mark.parametrize("recompute", [False, True])
def test_in_line_gives_the_bits_of_a_run_without_streams(nnb, b, s, recompute):
    g = torch.Generator().manual_seed(7)
    x, go = (torch.randn(s, b, 512, generator=g).cuda().bfloat16() for _ in range(2))
    got = []
    for use_streams in (True, False):
        cfg = _cfg(hidden_size=512, num_attention_heads=4, ffn_hidden_size=1024, num_layers=2, num_nanobatches=nnb,
                   use_streams=use_streams, checkpoint_activations=recompute)
        model = LayerStack(cfg, device="cuda", seed=3)
        assert cfg.nanobatches_in_line(s, b // nnb) is use_streams
        xd = x.clone().requires_grad_(True)
        for _ in range(2):                                                           # a second pass on the same model
            y = model(xd)
            y.backward(go)
        torch.cuda.synchronize()
        got.append([y.detach(), xd.grad] + [p.grad for p in model.parameters()])
    assert all(torch.equal(a, c) for a, c in zip(*got))


test_in_line_gives_the_bits_of_a_run_without_streams = gpu[0](gpu[1](test_in_line_gives_the_bits_of_a_run_without_streams))
