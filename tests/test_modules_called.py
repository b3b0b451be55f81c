"""What a program hangs on a module of the model - a hook, a subclass, another forward - runs, though the decoder computes most
modules' results inside launches of their neighbours."""
import pytest
import torch
import torch.nn as nn

import gptq_triton_amd as G
from gptq_triton_amd.llama import LlamaDecoderLayer, LlamaMLP, LlamaRMSNorm
from gptq_triton_amd.quant_linear import only_itself
from test_gpu_stream import random_quant_model
from test_loader import tiny_config

WIDE = dict(hidden_size=1024, num_attention_heads=8, intermediate_size=2816)  # widths the streaming order takes


def unfused_model(monkeypatch, seed, act_order=False):
    """A two-layer decoder whose gate and up are modules of their own, in streaming order."""
    monkeypatch.setattr(G, "make_fused_mlp", lambda model: None)
    model = random_quant_model(hidden=1024, inter=2816, heads=8, layers=2, groupsize=128, seed=seed, act_order=act_order)
    G.set_layout(model, "stream")
    return model


class Adapter(G.QuantLinear):
    """A projection that adds something to the product."""

    def forward(self, x):
        return super().forward(x) + 0.5


def hang(m, how, calls):
    """Make `m` do more than its class's forward.  Returns what undoes it."""
    if how == "forward hook":
        return m.register_forward_hook(lambda *_: calls.append(1)).remove
    if how == "pre hook":
        return m.register_forward_pre_hook(lambda *_: calls.append(1)).remove
    if how == "instance":
        real = m.forward
        m.forward = lambda *a, **k: calls.append(1) or real(*a, **k)
        return lambda: m.__dict__.pop("forward")
    if how == "global hook":
        return nn.modules.module.register_module_forward_hook(lambda mod, *_: calls.append(1) if mod is m else None).remove
    cls, real = type(m), type(m).forward
    if how == "class":
        cls.forward = lambda self, *a, **k: (calls.append(1) if self is m else None) or real(self, *a, **k)

        def undo():
            cls.forward = real
        return undo
    m.__class__ = type("Sub", (cls,), {"forward": lambda self, *a, **k: calls.append(1) or real(self, *a, **k)})

    def undo():
        m.__class__ = cls
    return undo


HOWS = ("forward hook", "pre hook", "instance", "global hook", "class", "subclass")


@pytest.mark.parametrize("how", HOWS)
def test_only_itself(how):
    q = G.QuantLinear(4, 128, 256, 256, bias=False)
    assert only_itself(q, G.QuantLinear) and not only_itself(nn.Linear(8, 8), G.QuantLinear) and not only_itself(len, G.QuantLinear)
    undo = hang(q, how, [])
    assert not only_itself(q, G.QuantLinear)
    undo()
    assert only_itself(q, G.QuantLinear)


def streamed_mlp(g_idx=False, mlp=None, **sizes):
    """An unfused MLP block whose gate and up look as in streaming order (no weights: nothing is launched)."""
    with torch.device("meta"):
        made = LlamaMLP(tiny_config(**(sizes or WIDE)))
    mlp = made if mlp is None else mlp
    for name in ("gate_proj", "up_proj", "down_proj"):
        old = getattr(made, name)
        with torch.device("meta"):
            q = G.QuantLinear(4, 128, old.in_features, old.out_features, bias=False, act_order=g_idx)
        q._stream_meta, q._stream_rows = torch.zeros(1, dtype=torch.int32), 16
        q._compact_perm = torch.arange(old.in_features, dtype=torch.int32) if g_idx else None
        setattr(mlp, name, q)
    return mlp


@pytest.mark.parametrize("how", HOWS)
@pytest.mark.parametrize("name", ["gate_proj", "up_proj"])
def test_gate_and_up_are_one_launch_only_while_nothing_hangs_on_them(name, how):
    mlp = streamed_mlp(g_idx=True)
    assert mlp._pair(2) is not None and mlp.input_order() is not None
    undo = hang(getattr(mlp, name), how, [])
    assert mlp._pair(2) is None and mlp.input_order() is None
    undo()
    assert mlp._pair(2) is not None
    undo = hang(mlp, how, [])
    assert mlp.input_order() is None and not mlp.norm_fusable(1)
    undo()
    assert mlp.input_order() is not None


@pytest.mark.parametrize("how", HOWS)
@pytest.mark.parametrize("act_order", [False, True])
def test_a_fused_mlp_is_called_while_something_hangs_on_it(how, act_order):
    """The decoder normalises inside the gate/up launch, and writes the norm in the order gate and up read, only where calling
    the block would do nothing else."""
    new = lambda k, n: G.QuantLinear(4, 128, k, n, bias=False, act_order=act_order)
    mlp = G.QuantLlamaMLP(new(1024, 2816), new(2816, 1024), new(1024, 2816))
    mlp._gate_meta, mlp._stream_rows = torch.zeros(1, dtype=torch.int32), 16   # (as in streaming order; nothing is launched)
    mlp._compact_rows = torch.arange(1024, dtype=torch.int32) if act_order else None
    fuses = lambda: [mlp.norm_fusable(rows) for rows in (1, 2, 4)]
    assert all(fuses()) and (mlp.input_order() is not None) == act_order
    undo = hang(mlp, how, [])
    assert not any(fuses()) and mlp.input_order() is None
    undo()
    assert all(fuses())


def test_the_pair_is_asked_for_the_projections_there_are():
    """Projections put in the place of narrower ones: the rows the launch takes are those of the new ones."""
    mlp = streamed_mlp()
    assert mlp._pair(16) is not None
    streamed_mlp(mlp=mlp, hidden_size=8192, num_attention_heads=64, intermediate_size=32768)
    assert mlp._pair(3) is not None and mlp._pair(4) is None and mlp._pair(16) is None
    streamed_mlp(mlp=mlp, **WIDE)
    assert mlp._pair(16) is not None


@pytest.mark.parametrize("how", HOWS)
def test_o_proj_is_called_while_something_hangs_on_it(how):
    q = G.QuantLinear(4, 128, 256, 768, bias=False)
    o = G.QuantLinear(4, 128, 256, 256, bias=False, act_order=True)
    o._compact_perm = torch.arange(256, dtype=torch.int32)
    attn = G.QuantLlamaAttention(tiny_config(), q, o)
    assert attn.context_order() is not None
    undo = hang(o, how, [])
    assert attn.context_order() is None
    undo()
    attn.o_proj = nn.Linear(256, 256, bias=False).half()          # any module
    x = torch.randn(1, 256).half()
    assert attn.context_order() is None and torch.equal(attn.project_out(x), attn.o_proj(x))


PLACES = {"layer": "", "norm 1": "input_layernorm", "norm 2": "post_attention_layernorm", "attention": "self_attn", "mlp": "mlp",
          "o": "self_attn.o_proj", "gate": "mlp.gate_proj", "up": "mlp.up_proj", "down": "mlp.down_proj"}


@pytest.mark.gpu
@pytest.mark.parametrize("act_order", [False, True])
@pytest.mark.parametrize("bsz,new", [(1, 1), (2, 1), (1, 7)])
def test_forward_runs_what_hangs_on_its_modules(monkeypatch, bsz, new, act_order):
    """Every way of hanging something on every module of a layer: it runs once per forward, and the logits stay those of the
    undisturbed model up to the rounding of the launches that are split for it."""
    model = unfused_model(monkeypatch, 51, act_order)
    torch.manual_seed(9)
    ids = torch.randint(0, model.config.vocab_size, (bsz, 6 + new)).cuda()
    _, past = model(ids[:, :6], use_cache=True)
    run = lambda: model(ids[:, 6:], past_key_values=past)[0].float()
    want = run()
    layer = model.model.layers[1]
    assert type(layer) is LlamaDecoderLayer
    modules = {k: layer.get_submodule(v) for k, v in PLACES.items()}
    modules["last norm"] = model.model.norm
    for where, m in modules.items():
        for how in HOWS:
            calls = []
            undo = hang(m, how, calls)
            got = run()
            undo()
            assert len(calls) == 1, (where, how, len(calls))
            assert (got - want).norm() <= 0.02 * want.norm(), (where, how)
    assert torch.equal(run(), want)


@pytest.mark.gpu
@pytest.mark.parametrize("act_order", [False, True])
@pytest.mark.parametrize("bsz", [1, 2, 4, 6])
def test_greedy_decoder_runs_what_hangs_on_a_fused_mlp(monkeypatch, bsz, act_order):
    """Once a step, with the block's own input and with what it makes of the output: the tokens are those of a decoder that calls
    its blocks in any case."""
    from gptq_triton_amd import decoder_ops
    model = random_quant_model(hidden=1024, inter=2816, heads=8, layers=2, groupsize=128, seed=54, act_order=act_order)
    ids = torch.randint(0, model.config.vocab_size, (bsz, 9), device="cuda", generator=torch.Generator(device="cuda").manual_seed(bsz))
    mlp = model.model.layers[1].mlp

    def tokens():
        dec = G.GreedyDecoder(model, bsz, 32)
        return torch.cat([dec.prefill(ids), dec.decode(5)], dim=1)

    plain = tokens()
    for how in HOWS:
        calls = []
        undo = hang(mlp, how, calls)
        tokens()
        undo()
        assert len(calls) == 1 + 5, (how, len(calls))
    turned = mlp.register_forward_hook(lambda m, args, out: -4 * out - args[0])
    got = tokens()
    with monkeypatch.context() as mp:
        mp.setattr(decoder_ops, "NORM_PAYS_ROWS", 0)
        want = tokens()
    turned.remove()
    assert torch.equal(got, want) and not torch.equal(got, plain)
    assert torch.equal(tokens(), plain)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["gate_proj", "up_proj", "down_proj", "o_proj"])
def test_adapters_add_to_the_product(monkeypatch, name):
    """A subclass of QuantLinear that adds a half to every output, in a forward pass of one token."""
    model = unfused_model(monkeypatch, 52)
    torch.manual_seed(10)
    ids = torch.randint(0, model.config.vocab_size, (1, 7)).cuda()
    _, past = model(ids[:, :6], use_cache=True)
    layer = model.model.layers[1]
    block = layer.self_attn if name == "o_proj" else layer.mlp
    run = lambda: model(ids[:, 6:], past_key_values=past)[0].float()
    plain = run()
    handle = getattr(block, name).register_forward_hook(lambda m, args, out: None)
    called = run()                       # the same launches as with the adapter
    handle.remove()
    getattr(block, name).__class__ = Adapter
    adapted = run()
    assert not torch.equal(adapted, called)
    # the same sum by a hook on an ordinary projection
    getattr(block, name).__class__ = G.QuantLinear
    handle = getattr(block, name).register_forward_hook(lambda m, args, out: out + 0.5)
    assert torch.equal(run(), adapted)
    handle.remove()
    assert torch.equal(run(), plain)


@pytest.mark.gpu
def test_another_norm_module(monkeypatch):
    """A norm with no variance_epsilon of its own."""
    class Norm(nn.Module):
        def __init__(self, old):
            super().__init__()
            self.old = old

        def forward(self, x):
            return self.old(x)

    model = unfused_model(monkeypatch, 53)
    ids = torch.arange(5).view(1, 5).cuda()
    want = model(ids)[0].float()
    model.model.layers[0].input_layernorm = Norm(model.model.layers[0].input_layernorm)
    assert isinstance(model.model.layers[0].input_layernorm.old, LlamaRMSNorm)
    got = model(ids)[0].float()
    assert (got - want).norm() <= 0.02 * want.norm()
