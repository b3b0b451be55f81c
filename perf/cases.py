"""Workloads for timing the package end to end: what a program that runs a 4-bit LLaMA on one GPU asks of it, through the
public entry points and with everything those calls do on the host included.

A case is a dict of plain values.  `kind` says which entry point it goes through:

  linear     QuantLinear.forward, or triton_matmul4 on a checkpoint's own tensors (`function`)
  mlp        QuantLlamaMLP.forward
  attention  QuantLlamaAttention.forward, a prompt or one token behind a key / value pair
  forward    LlamaForCausalLM.forward, logits and key / value pairs out (sampling loops, scoring)
  generate   GreedyDecoder.prefill and .decode, a request answered by a decoder that is kept

Shapes are the decoders of bench.py (LLaMA 7B, 13B with act-order, 30B) and, in draw(), generic widths between 1024 and
8192.  Decoder stacks are cut to a part of their layers, which are all alike, so that the inputs are made quickly.
Packed weights are uniform nibbles around zero points of 6 to 9, so that they have no mean of their own; scales are sized
so that a projection keeps the size of its input and the residual stream stays of order one through the stack, as a
trained model's does.
"""
from __future__ import annotations

import math

import torch

import gptq_triton_amd as G
from gptq_triton_amd.llama import LlamaRMSNorm

VOCAB = 32000
# (hidden, intermediate) of the decoders bench.py builds
SHAPES = ((4096, 11008), (5120, 13824), (6656, 17920))
GROUPS = (-1, 128, 512)


def listed():
    return [
        # one projection of a decode step, the smallest call there is (7B o_proj)
        {"name": "linear_1row", "kind": "linear", "function": False, "rows": 1, "k": 4096, "n": 4096, "groupsize": 128,
         "act_order": False, "bias": False, "layout": "stream"},
        # a program that keeps the checkpoint's tensors and calls the function, a few sequences at once (7B down_proj,
        # one group)
        {"name": "function_7rows", "kind": "linear", "function": True, "rows": 7, "k": 11008, "n": 4096, "groupsize": -1,
         "act_order": False, "bias": False, "layout": "checkpoint"},
        # a short prompt through one projection with all the options a checkpoint can have (13B o_proj)
        {"name": "linear_100rows", "kind": "linear", "function": False, "rows": 100, "k": 5120, "n": 5120, "groupsize": 128,
         "act_order": True, "bias": True, "layout": "stream"},
        # a long prompt through the widest projection (30B gate_proj)
        {"name": "function_2048rows", "kind": "linear", "function": True, "rows": 2048, "k": 6656, "n": 17920, "groupsize": 512,
         "act_order": False, "bias": False, "layout": "checkpoint"},
        # the MLP of a decode step, of a batch of sequences decoded together, and of a prompt of ordinary length
        {"name": "mlp_1row", "kind": "mlp", "rows": 1, "hidden": 4096, "inter": 11008, "groupsize": 128, "act_order": False,
         "layout": "stream"},
        {"name": "mlp_13rows", "kind": "mlp", "rows": 13, "hidden": 5120, "inter": 13824, "groupsize": 128, "act_order": True,
         "layout": "stream"},
        {"name": "mlp_500rows", "kind": "mlp", "rows": 500, "hidden": 4096, "inter": 11008, "groupsize": 128, "act_order": False,
         "layout": "stream"},
        # the attention block for one token behind 1500 others, and for a long prompt of odd length
        {"name": "attention_step", "kind": "attention", "batch": 1, "new": 1, "past": 1500, "hidden": 4096, "groupsize": -1,
         "act_order": False, "layout": "stream"},
        {"name": "attention_prompt", "kind": "attention", "batch": 1, "new": 1999, "past": 0, "hidden": 4096, "groupsize": -1,
         "act_order": False, "layout": "stream"},
        # one step of a sampling loop over two sequences, which needs the logits (a model as load_quant returns it: with
        # groups, gate and up stay separate)
        {"name": "forward_step", "kind": "forward", "batch": 2, "new": 1, "past": 333, "hidden": 4096, "inter": 11008, "layers": 8,
         "groupsize": 128, "act_order": False, "fuse_mlp": False, "layout": "stream"},
        # a request of 2000 prompt tokens and 48 answered ones, one captured graph a token
        {"name": "generate_1", "kind": "generate", "batch": 1, "prompt": 2000, "new": 48, "hidden": 4096, "inter": 11008, "layers": 16,
         "groupsize": 128, "act_order": False, "fuse_mlp": True, "graph": True},
        # eight short requests together, launched kernel by kernel (decode's default)
        {"name": "generate_8", "kind": "generate", "batch": 8, "prompt": 100, "new": 24, "hidden": 5120, "inter": 13824, "layers": 8,
         "groupsize": 128, "act_order": True, "fuse_mlp": True, "graph": False},
    ]


def _log_int(rng, low, high):
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high + 1))))))


def _widths(rng):
    if rng.random() < 0.5:
        return rng.choice(SHAPES)
    hidden = 256 * rng.randint(4, 32)
    return hidden, 256 * min(70, max(4, round(hidden * rng.uniform(2.5, 3.0) / 256)))  # at most the 30B decoder's


def _groupsize(rng, *ks):
    return rng.choice([g for g in GROUPS if g == -1 or all(k % g == 0 for k in ks)])


def draw(rng):
    kind = rng.choice(("linear", "linear", "mlp", "attention", "forward", "generate"))
    hidden, inter = _widths(rng)
    act_order = rng.random() < 0.25
    layout = "stream" if rng.random() < 0.75 else "checkpoint"
    if kind == "linear":
        k, n = rng.choice(((hidden, hidden), (hidden, 3 * hidden), (hidden, inter), (inter, hidden)))
        function = rng.random() < 0.4
        return {"kind": kind, "function": function, "rows": _log_int(rng, 1, 2048), "k": k, "n": n, "groupsize": _groupsize(rng, k),
                "act_order": act_order and not function, "bias": rng.random() < 0.25, "layout": "checkpoint" if function else layout}
    groupsize = _groupsize(rng, hidden, inter)
    act_order = act_order and groupsize != -1
    if kind == "mlp":
        return {"kind": kind, "rows": _log_int(rng, 1, 2048), "hidden": hidden, "inter": inter, "groupsize": groupsize,
                "act_order": act_order, "layout": layout}
    step = rng.random() < 0.5  # one token behind others, or a prompt
    batch = rng.choice((1, 1, 2, 4, 8))
    if kind == "attention":
        new, past = (1, _log_int(rng, 16, 2047)) if step else (_log_int(rng, 2, 2048 // batch), 0)
        return {"kind": kind, "batch": batch, "new": new, "past": past, "hidden": hidden, "groupsize": groupsize, "act_order": act_order,
                "layout": layout}
    fuse = groupsize == -1 or rng.random() < 0.5
    if kind == "forward":
        new, past = (1, _log_int(rng, 16, 2047)) if step else (_log_int(rng, 2, 1024 // batch), 0)
        return {"kind": kind, "batch": batch, "new": new, "past": past, "hidden": hidden, "inter": inter, "layers": rng.randint(2, 6),
                "groupsize": groupsize, "act_order": act_order, "fuse_mlp": fuse, "layout": layout}
    return {"kind": kind, "batch": batch, "prompt": _log_int(rng, 8, 2000 // batch), "new": rng.randint(8, 40), "hidden": hidden,
            "inter": inter, "layers": rng.randint(2, 6), "groupsize": groupsize, "act_order": act_order, "fuse_mlp": fuse,
            "graph": rng.random() < 0.5}


# ---- inputs ----------------------------------------------------------------------------------------------------------


class _Maker:
    """Random tensors on the GPU from one seed."""

    def __init__(self, seed):
        self.device = torch.device("cuda", torch.cuda.current_device())
        self.generator = torch.Generator(device=self.device)
        self.generator.manual_seed(seed)

    def words(self, shape):
        return torch.randint(-2 ** 31, 2 ** 31, shape, dtype=torch.int32, device=self.device, generator=self.generator)

    def normal(self, *shape):
        return torch.randn(shape, dtype=torch.float16, device=self.device, generator=self.generator)

    def fill(self, layer, gain=1.0, order=None):
        """Random contents of a QuantLinear whose output is about `gain` times as large as its input; order: the group of
        every input row (act-order), shared by projections that share their input."""
        layer.qweight.copy_(self.words(layer.qweight.shape))
        layer.qzeros.copy_((self.words(layer.qzeros.shape) & 0x33333333) + 0x55555555)  # stored, one less: 5 to 8
        spread = torch.rand(layer.scales.shape, device=self.device, generator=self.generator)
        layer.scales.copy_(gain * (0.7 + 0.6 * spread) / (4.75 * math.sqrt(layer.infeatures)))
        if layer.bias is not None:
            layer.bias.copy_(0.1 * self.normal(layer.outfeatures))
        if layer.g_idx is not None:
            layer.g_idx.copy_(order)

    def order(self, k, groupsize):
        if groupsize == -1:
            return torch.zeros(k, dtype=torch.int32, device=self.device)
        shuffled = torch.randperm(k, device=self.device, generator=self.generator)
        return (torch.arange(k, device=self.device) // groupsize)[shuffled].int()

    def linear(self, k, n, groupsize, act_order=False, bias=False, gain=1.0, order=None):
        with torch.device("meta"):
            layer = G.QuantLinear(4, groupsize, k, n, bias, act_order=act_order)
        layer = layer.to_empty(device=self.device)
        self.fill(layer, gain, order if order is not None or not act_order else self.order(k, groupsize))
        return layer


def _config(hidden, inter, layers, positions):
    cfg = G.LlamaConfigLite()
    cfg.hidden_size, cfg.intermediate_size, cfg.num_attention_heads = hidden, inter, hidden // 128
    cfg.num_hidden_layers, cfg.vocab_size, cfg.max_position_embeddings = layers, VOCAB, max(2048, positions)
    return cfg


def _settle(module, act_order, layout):
    """What load_quant does with a model once it is on the GPU."""
    holder = torch.nn.ModuleList([module])
    if act_order:
        G.quant_linear.compact_act_order(holder)
    if layout == "stream":
        G.set_layout(holder, "stream")
    return module


def _model(make, case, positions):
    cfg = _config(case["hidden"], case["inter"], case["layers"], positions)
    default = torch.get_default_dtype()
    torch.set_default_dtype(torch.half)
    try:
        with torch.device("meta"):
            model = G.LlamaForCausalLM(cfg)
            G.make_quant(model, 4, case["groupsize"], act_order=case["act_order"])
    finally:
        torch.set_default_dtype(default)
    model = model.to_empty(device=make.device)
    small = 1.0 / math.sqrt(2 * case["layers"])  # what a block adds to the residual stream
    for layer in model.model.layers:
        for names, gain in (("q_proj k_proj v_proj", 1.0), ("o_proj", small)):
            order = make.order(case["hidden"], case["groupsize"]) if case["act_order"] else None
            for name in names.split():
                make.fill(getattr(layer.self_attn, name), gain, order)
        for names, gain, k in (("gate_proj up_proj", 1.0, case["hidden"]), ("down_proj", small, case["inter"])):
            order = make.order(k, case["groupsize"]) if case["act_order"] else None
            for name in names.split():
                make.fill(getattr(layer.mlp, name), gain, order)
    for m in model.modules():
        if isinstance(m, LlamaRMSNorm):
            m.weight.copy_(1.0 + 0.1 * make.normal(case["hidden"]))
    # a trained model is fairly sure of the next token: here it is the one after the last
    embed = make.normal(VOCAB, case["hidden"])
    model.model.embed_tokens.weight.copy_(embed)
    model.lm_head.weight.copy_(0.05 * embed.roll(1, 0))
    G.make_quant_attn(model)
    if case["fuse_mlp"]:
        G.make_fused_mlp(model)
    return model


@torch.no_grad()
def prepare(case, seed):
    make = _Maker(seed)
    kind = case["kind"]
    if kind == "linear":
        layer = make.linear(case["k"], case["n"], case["groupsize"], case["act_order"], case["bias"])
        if not case["function"]:
            _settle(layer, case["act_order"], case["layout"])
        return {"case": case, "layer": layer, "x": make.normal(case["rows"], case["k"])}
    if kind == "mlp":
        hidden, inter, g, act = case["hidden"], case["inter"], case["groupsize"], case["act_order"]
        order = make.order(hidden, g) if act else None
        gate, up = (make.linear(hidden, inter, g, act, order=order) for _ in range(2))
        block = G.QuantLlamaMLP(gate, make.linear(inter, hidden, g, act), up)
        return {"case": case, "block": _settle(block, act, case["layout"]), "x": make.normal(case["rows"], hidden)}
    if kind == "attention":
        hidden, g, act = case["hidden"], case["groupsize"], case["act_order"]
        qkv, out = make.linear(hidden, 3 * hidden, g, act), make.linear(hidden, hidden, g, act)
        block = G.QuantLlamaAttention(_config(hidden, hidden, 1, case["past"] + case["new"]), qkv, out)
        shape = (case["batch"], hidden // 128, case["past"], 128)
        return {"case": case, "block": _settle(block, act, case["layout"]), "x": make.normal(case["batch"], case["new"], hidden),
                "past": (make.normal(*shape), make.normal(*shape)) if case["past"] else None}
    if kind == "forward":
        model = _settle(_model(make, case, case["past"] + case["new"]), case["act_order"], case["layout"])
        shape = (case["batch"], case["hidden"] // 128, case["past"], 128)
        past = [(make.normal(*shape), make.normal(*shape)) for _ in range(case["layers"])] if case["past"] else None
        ids = torch.randint(0, VOCAB, (case["batch"], case["new"]), device=make.device, generator=make.generator)
        return {"case": case, "model": model, "ids": ids, "past": past}
    model = _settle(_model(make, case, case["prompt"] + case["new"]), case["act_order"], "stream")
    ids = torch.randint(0, VOCAB, (case["batch"], case["prompt"]), device=make.device, generator=make.generator)
    return {"case": case, "decoder": G.GreedyDecoder(model, case["batch"], case["prompt"] + case["new"]), "ids": ids}


@torch.no_grad()
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        layer = state["layer"]
        if case["function"]:
            return G.triton_matmul4(layer.groupsize, state["x"], layer.qweight, layer.scales, layer.qzeros, layer.bias)
        return layer(state["x"])
    if kind == "mlp":
        return state["block"](state["x"])
    if kind == "attention":
        out, _, pair = state["block"](state["x"], past_key_value=state["past"], use_cache=True, causal=True)
        return out, pair
    if kind == "forward":
        return state["model"](state["ids"], past_key_values=state["past"], use_cache=True)
    decoder = state["decoder"]
    first = decoder.prefill(state["ids"])
    rest = decoder.decode(case["new"] - 1, use_graph=case["graph"])
    return {"first": first, "rest": rest, "caches": decoder.caches}


# ---- what a pass cannot do without, and how close another one comes ----------------------------------------------------


def _weights(k, n, groupsize):
    """Bytes of a packed projection."""
    groups = 1 if groupsize == -1 else k // groupsize
    return k * n // 2 + groups * (n // 2 + 2 * n)


def _projections(case):
    """(bytes, multiplications and additions a row) of one decoder layer's projections."""
    h, i, g = case["hidden"], case["inter"], case["groupsize"]
    return (_weights(h, 3 * h, g) + _weights(h, h, g) + 2 * _weights(h, i, g) + _weights(i, h, g), 2 * (4 * h * h + 3 * h * i))


def _attention_flops(batch, hidden, new, past):
    """Both products of causal attention: query j sees past + j + 1 rows."""
    return 4 * batch * hidden * (new * past + new * (new + 1) // 2)


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, k, n = case["rows"], case["k"], case["n"]
        return {"bytes": _weights(k, n, case["groupsize"]) + 2 * m * (k + n), "flops": 2 * m * k * n}
    g, h = case["groupsize"], case["hidden"]
    if kind == "mlp":
        m, i = case["rows"], case["inter"]
        return {"bytes": 2 * _weights(h, i, g) + _weights(i, h, g) + 4 * m * h, "flops": 6 * m * h * i}
    batch, new = case["batch"], case["new"]
    if kind == "attention":
        # the past is read, past and new rows are written to the pair that comes back
        past = case["past"]
        return {"bytes": _weights(h, 3 * h, g) + _weights(h, h, g) + 4 * batch * new * h + 4 * batch * h * (2 * past + new),
                "flops": 8 * batch * new * h * h + _attention_flops(batch, h, new, past)}
    per_layer, per_row = _projections(case)
    layers, head = case["layers"], 2 * VOCAB * h
    if kind == "forward":
        past = case["past"]
        return {"bytes": layers * (per_layer + 4 * batch * h * (2 * past + new)) + head + 2 * batch * new * (h + VOCAB),
                "flops": batch * new * (layers * per_row + 2 * h * VOCAB) + layers * _attention_flops(batch, h, new, past)}
    prompt, steps = case["prompt"], new - 1
    # every step reads the weights, the lm_head and the rows cached so far, and writes one row
    rows = steps * prompt + steps * (steps + 1) // 2
    return {"bytes": (steps + 1) * (layers * per_layer + head) + 4 * layers * batch * h * (prompt + steps + rows),
            "flops": batch * (prompt + steps) * layers * per_row + batch * (steps + 1) * 2 * h * VOCAB
            + layers * _attention_flops(batch, h, prompt + steps, 0)}


def tolerance(case):
    # fp16 results of fp32 sums: half a unit in the last place is 2.8e-4 in the 2-norm; one more rounding for every
    # intermediate result that is kept in fp16, and through a stack of layers they add up.  Tokens are whole numbers.
    return {"rel": {"linear": 1e-3, "mlp": 2e-3, "attention": 3e-3, "forward": 1e-2, "generate": 1e-2}[case["kind"]], "differ": 0.0}
