"""Operator sequences that run as one native call (operators/chains.py): found where the graph has them, bit for bit the
operators one by one, and left alone whenever something looks between the operators or replaced one."""

import dataclasses
import gc
import itertools
import threading
import weakref

import pytest
import torch

from kareus_amd import LayerConfig, LayerStack, operators
from kareus_amd.backend import get_backend
from kareus_amd.operators import PartitionableRMSNorm, ResidualForkOp, chains
from kareus_amd.partitions import Channel, ComputeOp, TensorPort, autograd_function
from kareus_amd.partitions.op_context import OperationContext
from kareus_amd.partitions.partition_base import PartitionBase
from kareus_amd.partitions.streams import stream_api


def config(nnb=1, **kw):
    base = dict(hidden_size=256, num_attention_heads=4, num_query_groups=2, kv_channels=64, ffn_hidden_size=320, num_layers=2,
                num_nanobatches=nnb, backend="hip")
    return LayerConfig(**{**base, **kw})


# ---- which sequences are found -------------------------------------------------------------------------------
@pytest.mark.parametrize("fuse", [True, False])
def test_every_segment_of_a_layer_is_a_chain(fuse):
    model = LayerStack(config(fuse_forward_epilogues=fuse), device="cpu")
    found = []
    for part in model.forward_partitions + model.backward_partitions:
        plans = part._plans()
        for i, chain in enumerate(part._op_chains):
            if isinstance(chain, (chains._ForwardChain, chains._BackwardChain)):
                assert [p.op_id for p in chain.plans] == [p.op_id for p in plans[i:i + chain.length]]
                found.append(type(chain).__name__)
    assert [found.count(n) for n in ("_ForwardAttention", "_ForwardMlp", "_BackwardMlp", "_BackwardAttention")] == [2, 2, 2, 2]


def test_a_model_is_freed_without_the_garbage_collector():
    """(A chain holds plans, and nothing of a plan or an operator holds the chain.)"""
    gc.collect()
    gc.disable()
    try:
        model = LayerStack(config(), device="cpu")
        for part in model.forward_partitions + model.backward_partitions:
            part._plans()
        weight = weakref.ref(model.layers[0].linear_qkv)
        del model, part
        assert weight() is None
    finally:
        gc.enable()


def test_a_subclass_or_another_order_is_no_chain():
    class Mine(PartitionableRMSNorm):
        pass

    model = LayerStack(config(), device="cpu")
    part = model.forward_partitions[0]
    part.comp_ops[1].operator = Mine(256, backend="hip")
    part._plans()
    assert not any(isinstance(c, chains._ForwardChain) for c in part._op_chains)


def with_a_reader(model, channels, layer=0):
    """The model's partitions built again with one more operator behind a layer's, which adds up two of the layer's channels."""
    class BiasDropoutAddOp(operators.BiasDropoutAddOp):   # (its name is what the overlap slots know)
        def get_input_channels(self):
            return [Channel(i, name) for i, name in enumerate(channels)]

        def get_output_channels(self):
            return [Channel(0, "sum")]

        def get_backward_ops(self):
            return []

        def fuser_forward(self, *a, **kw):
            got = super().fuser_forward(*a, **kw)
            self.sums.append(got[0])
            return got

    reader = BiasDropoutAddOp()
    reader.sums = []
    ops = model.layers[layer].get_all_operators() + [reader]
    model.layers[layer].get_all_operators = lambda: ops
    model._build_partitions()
    model.set_tensor_parallel_group(None)
    return reader


def found_in(partitions):
    names = []
    for part in partitions:
        part._plans()
        names += [type(c).__name__ for c in part._op_chains if isinstance(c, chains._Chain)]
    return names


@pytest.mark.parametrize("channels,left", [(("key", "value"), ["_ForwardMlp", "_ForwardAttention", "_ForwardMlp"]),
                                           (("residual", "main"), ["_ForwardAttention", "_ForwardMlp"] * 2),
                                           (("residual", "value"), ["_ForwardMlp", "_ForwardAttention", "_ForwardMlp"])])
def test_a_sequence_with_another_reader_inside_is_no_chain(channels, left):
    """The reader is in another partition than the tensors that it reads: key and value are made inside the attention sequence,
    the residual beside it."""
    model = LayerStack(config(), device="cpu")
    with_a_reader(model, channels)
    assert found_in(model.forward_partitions) == left


def test_a_reader_that_replaces_an_operator_or_reads_a_gradient_is_noticed():
    model = LayerStack(config(), device="cpu")
    part = model.forward_partitions[0]
    inside = part.comp_ops[3].get_output_tensor_ids()[1]       # the key in front of the rotary embedding
    assert found_in([part]) == ["_ForwardAttention"]
    part.comp_ops.append(ComputeOp(operators.BiasDropoutAddOp(), [TensorPort(0, inside), TensorPort(1, inside)],
                                   [TensorPort(0, "t_sum")], op_id=999))
    assert found_in([part]) == []
    behind = model.forward_partitions[1]                       # [residual add, fork, norm, ..]
    assert found_in([behind]) == ["_ForwardMlp"] and isinstance(behind._op_chains[0], chains._ForwardBehindAdd)
    handed_on = behind.comp_ops[0].get_output_tensor_ids()[0]
    behind.comp_ops.append(ComputeOp(operators.BiasDropoutAddOp(), [TensorPort(0, handed_on), TensorPort(1, "ext_main")],
                                     [TensorPort(0, "t_sum")], op_id=998))
    assert found_in([behind]) == ["_ForwardMlp"] and behind._op_chains[0] is None
    back = model.backward_partitions[0]
    assert found_in([back]) == ["_BackwardMlp"]
    known = back.read_twice
    back.read_twice, back._op_plans = known | {back.comp_ops[1].get_output_tensor_ids()[0]}, None
    assert found_in([back]) == []
    back.read_twice, back._op_plans = known, None
    assert found_in([back]) == ["_BackwardMlp"]
    back.read_twice = back._op_plans = None                   # nothing is known of the graph
    assert found_in([back]) == []


def test_a_second_thread_finds_no_plans_without_their_chains():
    """Two threads' first passes of one model: while one looks for chains, the other has to look for itself."""
    model = LayerStack(config(), device="cpu")
    part = model.forward_partitions[0]
    find, got = part._find_chains, []

    def first(plans):
        del part._find_chains
        other = threading.Thread(target=lambda: got.append((part._plans(), part._op_chains)))
        other.start()
        other.join()
        return find(plans)

    part._find_chains = first
    part._plans()
    (plans, chained), = got
    assert len(plans) == len(chained) and isinstance(chained[0], chains._ForwardAttention)


def test_a_second_thread_asks_for_every_backend_method(monkeypatch):
    """While one thread's first pass gathers what the backend's methods are, another's has to see all of them or none."""
    from kareus_amd.backend import hip

    seen, load = [], hip.load_native
    monkeypatch.setattr(chains, "_BACKEND_STOCK", type(chains._BACKEND_STOCK)())
    monkeypatch.setattr(hip, "load_native", lambda: seen.append(len(chains._BACKEND_STOCK)) or load())
    assert chains.chains_allowed()
    assert set(seen) == {0} and len(chains._BACKEND_STOCK) == len(chains._BACKEND_METHODS) + 1


def test_replaced_methods_are_noticed(monkeypatch):
    model = LayerStack(config(), device="cpu")
    ops = [p.operator for p in model.forward_partitions[0]._plans()]
    assert chains._untouched(ops)
    ops[2].fuser_forward = lambda *a, **k: None
    assert not chains._untouched(ops)
    del ops[2].fuser_forward
    ops[0]._backend_name = "eager"
    assert not chains._untouched(ops)
    del ops[0]._backend_name
    assert not chains._untouched(ops)
    ops[0]._backend_name = "hip"
    assert chains._untouched(ops)
    assert chains.chains_allowed()
    monkeypatch.setattr(ResidualForkOp, "fuser_forward", lambda *a, **k: None)
    assert not chains.chains_allowed()


class Halved(torch.nn.Module):
    def forward(self, w):
        return 0.5 * w


def test_an_operator_whose_class_changed_is_noticed():
    """(register_parametrization gives the module a class of its own, behind plans that are there.)"""
    model = LayerStack(config(), device="cpu")
    part = model.forward_partitions[0]
    ops = [p.operator for p in part._plans()]
    assert chains._untouched(ops)
    torch.nn.utils.parametrize.register_parametrization(model.layers[0].linear_qkv, "weight", Halved(), unsafe=True)
    assert not chains._untouched(ops) and found_in([part]) == ["_ForwardAttention"]


def test_a_replaced_backend_method_is_noticed(monkeypatch):
    from kareus_amd.backend import get_backend

    be = get_backend("hip")
    assert chains.chains_allowed()
    with monkeypatch.context() as m:
        m.setattr(type(be), "MAX_RUN_ROWS", 1)
        assert not chains.chains_allowed()
    with monkeypatch.context() as m:
        m.setitem(be.__dict__, "attn_fwd", lambda *a, **k: None)
        assert not chains.chains_allowed()
    for name in ("linear_wgrad_segments", "wgrad_segments_ok", "linear_wgrad"):   # (the sum over nanobatches in line)
        with monkeypatch.context() as m:
            m.setattr(type(be), name, lambda *a, **k: None)
            assert not chains.chains_allowed()
        with monkeypatch.context() as m:
            m.setitem(be.__dict__, name, lambda *a, **k: None)
            assert not chains.chains_allowed()
    with monkeypatch.context() as m:
        m.setattr(type(be), "MAX_WGRAD_SEGMENTS", 1)
        assert not chains.chains_allowed()
    with monkeypatch.context() as m:
        m.setattr(be, "_n", object())
        assert not chains.chains_allowed()
    assert chains.chains_allowed()


class HostBackend:
    """The two products that the weight gradient's sink needs, on the host."""
    class _n:
        wgrad_segments = staticmethod(lambda *a: None)

    linear_wgrad_segments = None
    _split_code = staticmethod(lambda split_k: 1)
    wgrad_segments_ok = staticmethod(lambda dys, xs: False)

    @staticmethod
    def linear_wgrad(dy, x, out=None, accumulate=False, split_k=True):
        dw = dy.t() @ x
        return dw if out is None else out.copy_(out + dw if accumulate else dw)


@pytest.mark.parametrize("order", [(0, 1, 2), (2, 0, 1)])
@pytest.mark.parametrize("ways", [way for way in itertools.product("co", repeat=3)])
def test_nanobatches_meet_in_the_sink_whichever_way_they_ran(ways, order):
    """One weight gradient over three nanobatches in line, each of which left its pair as a chain (c) or operator by operator (o)."""
    linear, be = operators.TERowParallelLinearOp(8, 16), HostBackend()
    sink = {"n": 3, "turn": [0], "defer": True, "pending": None, "in_line": True}
    pairs = [(torch.randn(4, 16), torch.randn(4, 8)) for _ in range(3)]
    got = []
    for i, way in zip(order, ways):
        ctx = OperationContext()
        ctx.wgrad_sink, ctx.nanobatch_index, ctx.alone = sink, i, True
        got.append(chains._add_pair(be, linear, ctx, *pairs[i]) if way == "c" else linear._weight_grad(be, ctx, *pairs[i]))
    want = pairs[0][0].t() @ pairs[0][1]
    for dy, x in pairs[1:]:
        want = want + dy.t() @ x
    assert got[0] is None and got[1] is None and torch.equal(got[2], want) and sink["turn"] == [1] and sink["pairs"] is None


# ---- the same bits ---------------------------------------------------------------------------------------------------
def run(cfg, s, b, *, seed=0, grad=True, before=None, hooks=None):
    torch.manual_seed(seed)
    model = LayerStack(cfg, device="cuda", seed=3)
    if before is not None:
        before(model)
    x = torch.randn(s, b, cfg.hidden_size, generator=torch.Generator().manual_seed(1)).to("cuda", torch.bfloat16)
    go = torch.randn(s, b, cfg.hidden_size, generator=torch.Generator().manual_seed(2)).to("cuda", torch.bfloat16)
    if not grad:
        with torch.no_grad():
            return [model(x)]
    x.requires_grad_(True)
    out = []
    for _ in range(2):   # (the second pass on gradients and plans that are there)
        with (hooks() if hooks is not None else torch.enable_grad()):
            y = model(x)
        y.backward(go)
        out.append(y.detach())
    torch.cuda.synchronize()
    return out + [x.grad] + [p.grad for p in model.parameters()]


def both(monkeypatch, *args, **kw):
    """The pass with chains, which have to have run (``ran``: how many of each), and the pass without."""
    ran = {}
    with monkeypatch.context() as m:
        for cls in (chains._ForwardAttention, chains._ForwardMlp, chains._BackwardMlp, chains._BackwardAttention):
            def watched(self, *a, _run=cls.run, _name=cls.__name__):
                got = _run(self, *a)
                ran[_name] = ran.get(_name, 0) + (got is not None and got is not False)
                return got
            m.setattr(cls, "run", watched)
        got = run(*args, **kw)
    with monkeypatch.context() as m:
        m.setattr(autograd_function, "_chains", lambda config: False)
        want = run(*args, **kw)
    assert len(got) == len(want)
    for a, b in zip(got, want):
        assert (a is None) == (b is None) and (a is None or torch.equal(a, b))
    return ran


CASES = {
    "one nanobatch": (config(), 128, 2),
    "odd sizes": (config(), 104, 3),
    "heads of 128, one group, one head": (config(num_attention_heads=1, num_query_groups=1, kv_channels=128), 72, 1),
    "no epilogue fusion": (config(fuse_forward_epilogues=False), 96, 2),
    "activation of its own": (config(ffn_hidden_size=344), 96, 2),          # no SwiGLU epilogue for this width
    "per-head norms and dropout": (config(qk_layernorm=True, hidden_dropout=0.2), 96, 2),
    "recomputation": (config(checkpoint_activations=True, hidden_dropout=0.1), 96, 2),
    "nanobatches in line": (config(2), 96, 4),
    "nanobatches in line, tokens no multiple of 64": (config(2, qk_layernorm=True), 104, 2),
    "four nanobatches in line, recomputed": (config(4, checkpoint_activations=True), 64, 4),
    "nanobatches on one stream": (config(2, use_streams=False), 96, 4),
    "accumulated weight gradients": (config(2, wgrad_over_all_nanobatches=False), 96, 4),
    "gradients summed by autograd": (config(2, fuse_wgrad_accumulation=False), 96, 4),
    "nanobatches on streams": (config(2, in_line_below_ms=0.0), 96, 4),
}


@pytest.mark.parametrize("what", sorted(CASES))
@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a HIP device")
def test_a_chain_has_the_bits_of_its_operators(what, monkeypatch):
    cfg, s, b = CASES[what]
    ran = both(monkeypatch, cfg, s, b)
    passes = 2 * cfg.num_layers * cfg.num_nanobatches
    again = 2 if cfg.checkpoint_activations else 1
    assert ran["_ForwardAttention"] == ran["_ForwardMlp"] == passes * again
    if what != "no epilogue fusion":
        assert ran["_BackwardAttention"] == ran["_BackwardMlp"] == passes


ON_STREAMS = {
    "two": (config(2), 96, 4),
    "two, tokens no multiple of 64, per-head norms, dropout": (config(2, qk_layernorm=True, hidden_dropout=0.2), 104, 2),
    "four, weight gradients at the end": (config(4), 64, 4),                # (their launches are left to the end of the pass)
    "four, weight gradients at once": (config(4, wgrad_launches_at_end=False), 64, 4),
    "accumulated weight gradients": (config(2, wgrad_over_all_nanobatches=False), 96, 4),
    "gradients summed by autograd": (config(2, fuse_wgrad_accumulation=False), 96, 4),
    "recomputation": (config(2, checkpoint_activations=True), 96, 4),
}


@pytest.mark.parametrize("what", sorted(ON_STREAMS))
@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a HIP device")
def test_backward_chains_of_nanobatches_on_streams(what, monkeypatch):
    """Every nanobatch's backward chains run on its own stream; the operands of the weight gradients meet in the layer's sink with
    the events behind them."""
    cfg, s, b = ON_STREAMS[what]
    cfg = dataclasses.replace(cfg, in_line_below_ms=0.0)
    ran = both(monkeypatch, cfg, s, b)
    assert ran["_BackwardAttention"] == ran["_BackwardMlp"] == 2 * cfg.num_layers * cfg.num_nanobatches


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a HIP device")
def test_the_first_projection_of_a_chain_leaves_its_event_before_the_other_steps(monkeypatch):
    """Nanobatches on streams: the operands of the out-projection's and of fc2's weight gradient are left, with their event, inside
    the native call, as the operators would leave them; an error there leaves the call."""
    log, api, native = [], stream_api(), get_backend("hip")._n
    new_event = api.new_event

    def event(*a):
        log.append("event")
        return new_event(*a)

    monkeypatch.setattr(api, "new_event", event)
    for name in ("mlp_chain_bwd", "attn_chain_bwd"):
        def call(*a, _call=getattr(native, name)):
            log.append("in")
            got = _call(*a)
            log.append("out")
            return got
        monkeypatch.setattr(native, name, call)
    cfg = dataclasses.replace(config(2), in_line_below_ms=0.0)
    run(cfg, 96, 4)
    starts = [i for i, what in enumerate(log) if what == "in"]
    assert len(starts) == 2 * 2 * cfg.num_layers * cfg.num_nanobatches
    assert all(log[i + 1:i + 3] == ["event", "out"] for i in starts)

    def no_event(*a):
        if log[-1] == "in":
            raise RuntimeError("no event")
        return event(*a)

    monkeypatch.setattr(api, "new_event", no_event)
    with pytest.raises(RuntimeError, match="no event"):
        run(cfg, 96, 4)
    torch.cuda.synchronize()


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a HIP device")
def test_chains_without_gradients_and_under_saved_tensor_hooks(monkeypatch):
    ran = both(monkeypatch, config(2), 96, 4, grad=False)
    assert ran["_ForwardAttention"] == 4
    both(monkeypatch, config(), 96, 2, hooks=lambda: torch.autograd.graph.save_on_cpu())
    seen = []
    both(monkeypatch, config(), 96, 2, hooks=lambda: torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(t.shape) or t,
                                                                                              lambda t: t))
    half = len(seen) // 2
    assert half and seen[:half] == seen[half:]     # the same tensors in the same order


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a HIP device")
def test_a_saved_attention_output_with_gaps_runs_operator_by_operator(monkeypatch):
    """(The native backward reads it dense; the answer comes before anything is launched.)"""
    def with_gaps(t):
        if t.shape != (96, 2, 4, 64):
            return t
        gaps.append(torch.empty(96, 2, 4, 128, dtype=t.dtype, device=t.device)[..., :64].copy_(t))
        return gaps[-1]

    gaps = []
    ran = both(monkeypatch, config(), 96, 2, hooks=lambda: torch.autograd.graph.saved_tensors_hooks(lambda t: t, with_gaps))
    assert gaps and ran.get("_BackwardAttention", 0) == 0 and ran["_BackwardMlp"] == 4


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a HIP device")
def test_a_tensor_inside_a_sequence_is_there_for_its_other_reader(monkeypatch):
    """An operator behind the layer reads the first layer's key and value; the block's output may be any channel."""
    sums = []
    both(monkeypatch, config(2), 96, 4, before=lambda model: sums.append(with_a_reader(model, ("key", "value")).sums))
    assert len(sums[0]) == len(sums[1]) == 4 and all(torch.equal(a, b) for a, b in zip(*sums))
    both(monkeypatch, config(num_layers=1), 96, 2, grad=False,
         before=lambda model: setattr(model, "seed_config", dataclasses.replace(model.seed_config, fwd_output_channel="value")))


@pytest.mark.parametrize("which", [0, 1])
@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a HIP device")
def test_one_of_two_nanobatches_in_line_runs_operator_by_operator(which, monkeypatch):
    """The saved attention outputs of one nanobatch come back with gaps: its attention runs one by one, the other's as a chain, and
    the two meet in the projections' weight gradients."""
    def hooks():
        seen = []

        def pack(t):
            if t.shape != (96, 2, 4, 64):
                return t
            seen.append(t)
            return t if (len(seen) - 1) // 2 != which else torch.empty(96, 2, 4, 128, dtype=t.dtype, device=t.device)[..., :64].copy_(t)
        return torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t)

    ran = both(monkeypatch, config(2), 96, 4, hooks=hooks)
    assert ran["_BackwardAttention"] == 4 and ran["_BackwardMlp"] == 8


def misaligned(t):
    """A dense copy two bytes beyond a boundary of 16: the library turns it down before it launches anything."""
    return torch.empty(t.numel() + 8, dtype=t.dtype, device=t.device)[1:t.numel() + 1].view(t.shape).copy_(t)


@pytest.mark.parametrize("where", ["linear_qkv", "linear_proj", "linear_fc1", "linear_fc2", "q_layernorm", "dgrad linear_qkv",
                                   "dgrad linear_proj", "dgrad linear_fc1", "dgrad linear_fc2", "wgrad (192, 320)", "wgrad (192, 256)",
                                   "head dimension"])
@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a HIP device")
def test_a_call_that_fails_is_named_as_by_its_operator(where, monkeypatch):
    """The same error, with the call's sizes, from a sequence and from its operators."""
    def broken():
        cfg = config(num_layers=1, qk_layernorm=True, kv_channels=136 if where == "head dimension" else 64)
        model = LayerStack(cfg, device="cuda", seed=3)
        layer = model.layers[0]
        x = torch.randn(96, 2, 256, device="cuda").bfloat16().requires_grad_(True)
        weight = {"q_layernorm": lambda: layer.qkv_postprocess.q_layernorm}.get(where, lambda: getattr(layer, where.split()[-1], None))()
        hooks = torch.autograd.graph.saved_tensors_hooks(
            lambda t: t, lambda t: misaligned(t) if where == f"wgrad {tuple(t.shape)}" else t)
        with pytest.raises(RuntimeError) as failure:
            if weight is not None and not where.startswith("dgrad"):
                weight.weight.data = misaligned(weight.weight.data)
            with hooks:
                y = model(x)
            if weight is not None:
                weight.weight.data = misaligned(weight.weight.data)
            y.sum().backward()
        torch.cuda.synchronize()
        return str(failure.value)

    chained = broken()
    with monkeypatch.context() as m:
        m.setattr(autograd_function, "_chains", lambda config: False)
        assert chained == broken()
    assert "(code -" in chained
    if "grad" in where or where.startswith("linear"):
        assert "M=" in chained and f"layout={2 if 'wgrad' in where else 1 if 'dgrad' in where else 0}" in chained


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a HIP device")
def test_a_parametrized_weight_runs_operator_by_operator(monkeypatch):
    """Registered on a model that has run: its layer leaves the chains, and the product is that of the weight it now has."""
    x = torch.randn(96, 2, 256, generator=torch.Generator().manual_seed(1)).to("cuda", torch.bfloat16)
    model, plain = (LayerStack(config(), device="cuda", seed=3) for _ in range(2))
    with torch.no_grad():
        first = model(x)
        torch.nn.utils.parametrize.register_parametrization(model.layers[0].linear_qkv, "weight", Halved(), unsafe=True)
        plain.layers[0].linear_qkv.weight.mul_(0.5)
        got, want = model(x), plain(x)
    assert torch.equal(got, want) and not torch.equal(got, first)


@pytest.mark.parametrize("part", ["linear_fc1", "linear_proj", "pre_mlp_layernorm"])
@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a HIP device")
def test_a_frozen_weight_gets_no_gradient(part, monkeypatch):
    both(monkeypatch, config(), 96, 2, before=lambda model: getattr(model.layers[1], part).weight.requires_grad_(False))


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a HIP device")
def test_an_operator_or_a_timer_between_the_operators_is_served(monkeypatch):
    """A method replaced on one operator runs; a timer sees every operator."""
    calls, model = [], LayerStack(config(), device="cuda", seed=3)
    rope = model.layers[0].rotary
    inner = rope.fuser_forward
    rope.fuser_forward = lambda *a, **k: calls.append("rope") or inner(*a, **k)
    x = torch.randn(96, 2, 256, device="cuda").bfloat16()
    with torch.no_grad():
        y = model(x)
        assert calls == ["rope"]
        del rope.fuser_forward
        assert torch.equal(model(x), y) and calls == ["rope"]

        class Timer:
            def begin(self, part): calls.append("begin")
            def end(self, part): calls.append("end")
            def op_done(self, part, idx): calls.append(idx)
        monkeypatch.setattr(PartitionBase, "timer", Timer())
        calls.clear()
        assert torch.equal(model(x), y)
    assert [c for c in calls if not isinstance(c, str)] == list(range(7)) + list(range(6)) + list(range(8)) + list(range(6)) + [0]
    assert calls.count("begin") == calls.count("end") == 5
