"""What a user has this framework compute: training steps and forward passes of decoder-layer stacks through
``LayerStack`` and ``GPTModelShard``, over the sizes, options and layouts that the repository's configurations
and benchmark name.

A case is a flat dict:
  h, nq, nkv, hd, ffn    one GPU's shard of a decoder layer (heads and FFN columns are per-shard counts)
  layers, b, s           stack depth, sequences, tokens per sequence
  nnb                    nanobatches (each on a stream of its own when there are several)
  kind                   "step"     forward + backward of the stack, hidden states in, gradients out
                         "loss"     token ids -> mean loss -> backward through embedding, stack and output layer
                         "logits"   token ids -> logits without gradients
  recompute              activation checkpointing
  qk_norm, dropout       per-head query / key norms, hidden dropout probability
  vocab                  rows of the vocabulary shard ("loss" and "logits")
  plan                   file of kareus_amd/plans that schedules the step ("" for none)
"""

from __future__ import annotations

import math

import torch

from kareus_amd import LayerConfig, LayerStack
from kareus_amd.model import GPTModelShard
from kareus_amd.plans import plan_path
from kareus_amd.scheduler import PipelineCommScheduler
from kareus_amd.scheduler.parser import parse_schedule_file

#: Shard shapes of the repository's workloads: (hidden, query heads, KV heads, head dim, FFN columns).
SHARDS = {
    "small": dict(h=512, nq=8, nkv=8, hd=64, ffn=1376, qk_norm=False, dropout=0.0, vocab=4096),
    "1b": dict(h=2048, nq=32, nkv=8, hd=64, ffn=8192, qk_norm=False, dropout=0.0, vocab=32064),
    "3b tp8": dict(h=3072, nq=3, nkv=1, hd=128, ffn=1024, qk_norm=False, dropout=0.0, vocab=16384),
    "3b": dict(h=3072, nq=24, nkv=8, hd=128, ffn=8192, qk_norm=False, dropout=0.0, vocab=32064),
    "8b tp4": dict(h=4096, nq=8, nkv=2, hd=128, ffn=3584, qk_norm=False, dropout=0.0, vocab=32064),
    "8b": dict(h=4096, nq=32, nkv=8, hd=128, ffn=14336, qk_norm=False, dropout=0.0, vocab=32064),
    "qwen3 tp8": dict(h=2048, nq=2, nkv=1, hd=128, ffn=768, qk_norm=True, dropout=0.1, vocab=16384),
}


def _case(shard, b, s, nnb, *, layers=1, kind="step", recompute=False, plan="", name=None):
    c = dict(SHARDS[shard], b=b, s=s, nnb=nnb, layers=layers, kind=kind, recompute=recompute, plan=plan)
    if kind == "step":
        c["vocab"] = 0
    return dict(c, name=name) if name else c


def listed():
    return [
        # a small layer with heads of 64, two nanobatches: unit-test sized models, all launches and host work
        _case("small", 2, 256, 2, name="small_step"),
        # one short sequence on a large model's shard: fine-tuning on short samples
        _case("8b tp4", 1, 512, 1, name="8b_tp4_short_step"),
        # scoring one prompt of an odd length, no gradients
        _case("8b tp4", 1, 776, 1, layers=2, kind="logits", name="8b_tp4_prompt_logits"),
        # three packed sequences of a length that no tile divides
        _case("8b tp4", 3, 2008, 1, name="8b_tp4_ragged_step"),
        # token ids to weight gradients, with activation checkpointing
        _case("8b tp4", 2, 2048, 1, kind="loss", recompute=True, name="8b_tp4_loss_recompute"),
        # the thin shard of an eight-way tensor-parallel 3B layer, two nanobatches of four sequences
        _case("3b tp8", 8, 4096, 2, name="3b_tp8_step"),
        # eight-way shard with per-head norms and hidden dropout
        _case("qwen3 tp8", 8, 4096, 2, name="qwen3_tp8_step"),
        # a full-width layer with heads of 64
        _case("1b", 2, 4096, 1, name="1b_step"),
        # the four-way shard of an 8B layer: as four nanobatches on their streams, and in one piece
        _case("8b tp4", 4, 4096, 4, name="8b_tp4_step_4nb"),
        _case("8b tp4", 4, 4096, 1, name="8b_tp4_step"),
        # a full-width 3B layer
        _case("3b", 4, 4096, 1, name="3b_step"),
        # four full-width 8B layers at 8192 tokens under a per-microbatch plan
        _case("8b", 2, 8192, 2, layers=4, plan="llama31_8b_4layers_mbs2_seq8192.py", name="8b_stack_step"),
    ]


def draw(rng):
    """One more case: any shard, sequence lengths over 96..8192 (a nanobatch's tokens are a multiple of 8, as the
    kernels ask; a third of the lengths are whole tiles), 1 to 8 sequences, one or two layers (one under a loss),
    all three kinds, at most the largest listed case's work."""
    most = max(work(c)["flops"] for c in listed())
    while True:
        shard = rng.choice(sorted(SHARDS))
        s = int(round(math.exp(rng.uniform(math.log(96), math.log(8192)))))
        b = rng.choice((1, 2, 3, 4, 6, 8))
        nnb = rng.choice([n for n in (1, 2, 4) if b % n == 0])
        unit = 128 if rng.random() < 0.35 else 8 // math.gcd(b // nnb, 8)
        s = max(unit, s // unit * unit)
        if b * s > 32768:
            continue
        kind = rng.choice(("step", "step", "step", "loss", "logits"))
        c = _case(shard, b, s, nnb, layers=1 if kind == "loss" else rng.choice((1, 1, 2)), kind=kind,
                  recompute=kind != "logits" and rng.random() < 0.2)
        if work(c)["flops"] <= most:
            return c


def _config(c):
    return LayerConfig(hidden_size=c["h"], num_attention_heads=c["nq"], num_query_groups=c["nkv"], kv_channels=c["hd"],
                       ffn_hidden_size=c["ffn"], num_layers=c["layers"], num_nanobatches=c["nnb"], backend="hip",
                       checkpoint_activations=c["recompute"], hidden_dropout=c["dropout"], qk_layernorm=c["qk_norm"])


def prepare(case, seed):
    """The model with its weights, and one batch: hidden states and an upstream gradient N(0, 1), or token ids and
    labels.  Weights N(0, 0.02) drawn on the device (the modules draw on the default device)."""
    c = case
    cfg = _config(c)
    if c["plan"] and c["nnb"] > 1:
        path = plan_path(c["plan"])
        cfg.kareus_scheduler = PipelineCommScheduler(path, pp_rank=0,
                                                     num_microbatches=len(parse_schedule_file(path, False, False)[0]))
    torch.manual_seed(seed)
    with torch.device("cuda"):
        if c["kind"] == "step":
            model = LayerStack(cfg, device="cuda")
            x = torch.randn(c["s"], c["b"], c["h"]).bfloat16().requires_grad_(True)
            go = torch.randn(c["s"], c["b"], c["h"]).bfloat16()
            data = (x, go)
        else:
            model = GPTModelShard(cfg, vocab_rows=c["vocab"], device="cuda")
            data = tuple(torch.randint(0, c["vocab"], (c["b"], c["s"])) for _ in range(2))
    return dict(model=model, named=list(model.named_parameters()), data=data, kind=c["kind"], seed=seed,
                dropout=c["dropout"] > 0.0, scheduler=cfg.kareus_scheduler, left=0)


def run(state):
    """One pass.  A step returns the output and every gradient, a loss pass the per-token losses and every
    gradient, a logits pass the logits."""
    model = state["model"]
    if state["dropout"]:
        torch.default_generator.manual_seed(state["seed"])  # the program's own seed for its dropout masks
    if state["kind"] == "logits":
        with torch.no_grad():
            return {"logits": model(state["data"][0])}
    for _, p in state["named"]:
        p.grad = None
    sch = state["scheduler"]
    if sch is not None:  # each pass is one microbatch of the plan, which starts over when it is used up
        if state["left"] == 0:
            sch.on_step_begin()
            state["left"] = len(sch._schedule_items)
        sch.on_instruction_begin("forward")
    if state["kind"] == "step":
        x, go = state["data"]
        x.grad = None
        out = model(x)
        if sch is not None:
            sch.on_instruction_end("forward")
            sch.on_instruction_begin("backward")
        out.backward(go)
        if sch is not None:
            sch.on_instruction_end("backward")
            state["left"] -= 1
            if state["left"] == 0:
                sch.on_step_end()
        got = {"out": out.detach(), "dx": x.grad}
    else:
        ids, labels = state["data"]
        loss = model(ids, labels)
        loss.mean().backward()
        got = {"loss": loss.detach()}
    for name, p in state["named"]:
        got[name] = p.grad
    return got


def work(case):
    """Weights, inputs, outputs and gradients once each (bf16); the products of the layers and of the output layer
    (backward twice the forward) and causal attention (backward 2.5 times the forward).  Recomputed activations
    do not count."""
    c = case
    t = c["b"] * c["s"]
    qkv = (c["nq"] + 2 * c["nkv"]) * c["hd"]
    weights = c["layers"] * (c["h"] * (qkv + c["nq"] * c["hd"] + 3 * c["ffn"] + 2) + (2 * c["hd"] if c["qk_norm"] else 0))
    gemm = 2 * t * c["layers"] * c["h"] * (qkv + c["nq"] * c["hd"] + 3 * c["ffn"])
    attn = 2 * c["layers"] * c["b"] * c["nq"] * c["s"] ** 2 * c["hd"]
    if c["kind"] == "step":
        return {"bytes": 2 * (4 * t * c["h"] + 2 * weights), "flops": 3 * gemm + 3.5 * attn}
    head = c["vocab"] * c["h"]
    if c["kind"] == "logits":
        return {"bytes": 8 * t + 2 * (weights + head + min(t, c["vocab"]) * c["h"] + t * c["vocab"]),
                "flops": gemm + attn + 2 * t * head}
    return {"bytes": 20 * t + 2 * (2 * weights + 2 * head + min(t, c["vocab"]) * c["h"] + head),
            "flops": 3 * gemm + 3.5 * attn + 6 * t * head}


def tolerance(case):
    """bf16 results with fp32 sums.  Measured on this path against itself with its contractions summed in another
    order (uncut GEMMs, the attention kernels' other form), worst output of 52 cases: one layer 6.0e-3 of the norm and
    0.048 of the root mean square, two layers 1.4e-2 and 0.12 (every layer rounds activations and gradients to bf16
    again, and the attention gradients behind a random-weight layer are small differences), logits 1.0e-2 and 0.064,
    behind a loss 7.6e-3 and 0.25, in the embedding's gradient, whose rows are sums of a few tokens: four times that,
    and at most 3e-2."""
    if case["kind"] == "loss":
        return {"rel": 3e-2, "max": 0.99}
    if case["kind"] == "logits" or case["layers"] > 1:
        return {"rel": 3e-2, "max": 0.48}
    return {"rel": 2.4e-2, "max": 0.2}
