"""Quantised modules whose tensors a loader holds as parameters, or as plain attributes, instead of buffers."""
import pytest
import torch
import torch.nn as nn

import gptq_triton_amd as G
from gptq_triton_amd.quant_linear import child, compact_act_order
from test_gpu_stream import random_quant_model


def as_parameters(m):
    for name, t in list(m._buffers.items()):
        if t is not None:
            del m._buffers[name]
            m.register_parameter(name, nn.Parameter(t, requires_grad=False))


def as_attributes(m):
    for name, t in list(m._buffers.items()):
        del m._buffers[name]
        object.__setattr__(m, name, t)


FORMS = [as_parameters, as_attributes]


def streamed(m, names):
    for name in names:
        setattr(m, name, torch.zeros(1, dtype=torch.int32))
    m._stream_rows = 16
    return m


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("stream", [False, True])
def test_the_tensors_are_found(form, stream):
    q = G.QuantLinear(4, 128, 1024, 1024, bias=True, act_order=True)
    q.bias.zero_()
    q._compact_perm = torch.arange(1024, dtype=torch.int32)
    if stream:
        streamed(q, ["_stream_meta"])
    tensors = {n: t for n, t in q._buffers.items() if t is not None}
    form(q)
    assert q.bias_tensor() is not None and torch.equal(q.bias_tensor(), tensors["bias"])
    assert torch.equal(q.row_permutation(), tensors["_compact_perm"])
    words = q.stream_weights(1)
    assert (words is None) == (not stream)
    if stream:
        assert torch.equal(words[0], tensors["qweight"]) and torch.equal(words[1], tensors["_stream_meta"])
    with pytest.raises(RuntimeError, match="GPU"):     # off the GPU: refused for that, and for nothing else
        q(torch.zeros(1, 1024, dtype=torch.float16))


@pytest.mark.gpu
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("layout", ["checkpoint", "stream"])
@pytest.mark.parametrize("act_order", [False, True])
def test_the_same_results(form, layout, act_order):
    model = random_quant_model(hidden=1024, inter=2816, heads=8, layers=1, groupsize=128, seed=71, act_order=act_order)
    layer = model.model.layers[0]
    compact_act_order(model)
    G.set_layout(model, layout)
    x1, x20 = torch.randn((1, 1, 1024), device="cuda").half(), torch.randn((1, 20, 1024), device="cuda").half()
    run = lambda: [m(x) for x in (x1, x20) for m in (layer.mlp, layer.self_attn.o_proj)] + [layer.self_attn(hidden_states=x)[0] for x in (x1, x20)]
    want = run()
    for m in (layer.mlp, layer.mlp.down_proj, layer.self_attn.o_proj, layer.self_attn.qkv_proj):
        form(m)
    for a, b in zip(run(), want):
        assert torch.equal(a, b)


def test_submodules_are_found_where_they_are_held():
    m, sub = nn.Module(), nn.Identity()
    m.registered = sub
    object.__setattr__(m, "plain", sub)
    assert child(m, "registered") is sub and child(m, "plain") is sub
    with pytest.raises(AttributeError):
        child(m, "none")
