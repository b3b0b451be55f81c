"""The inverse row permutations that producers write by: worked out again for every other permutation, wherever its memory lies."""
import weakref

import pytest
import torch

import gptq_triton_amd as G
from gptq_triton_amd.quant_linear import inverse_permutation
from test_gpu_stream import random_quant_model
from test_loader import tiny_config

K = 4096


def attention():
    q = G.QuantLinear(4, 128, K, 3 * K, bias=False, act_order=True)
    o = G.QuantLinear(4, 128, K, K, bias=False, act_order=True)
    attn = G.QuantLlamaAttention(tiny_config(hidden_size=K, num_attention_heads=32), q, o)
    return attn, {"context": (o, attn.context_order), "input": (q, attn.input_order)}


@pytest.mark.parametrize("which", ["context", "input"])
def test_a_permutation_lives_as_long_as_its_inverse_is_kept(which):
    """Its address names the kept inverse: given back, the memory could hold the next permutation, and that one be taken for it."""
    attn, ways = attention()
    q, order = ways[which]
    values = [torch.randperm(K).int() for _ in range(2)]
    q._compact_perm = values[0].clone()
    old = weakref.ref(q._compact_perm)
    assert torch.equal(order(), inverse_permutation(values[0])) and order() is order()
    q._compact_perm = None                        # (as load_state_dict() does to a compacted module)
    assert old() is not None
    q._compact_perm = values[1].clone()
    assert torch.equal(order(), inverse_permutation(values[1]))
    assert old() is None                          # one permutation is kept, not all there were


@pytest.mark.parametrize("which", ["context", "input"])
def test_a_permutation_of_inference_mode_leaves_the_gather_to_the_projection(which):
    """An act-order module works out its permutation in the first call; in inference mode that is a tensor without a version."""
    attn, ways = attention()
    q, order = ways[which]
    with torch.inference_mode():
        q._compact_perm = torch.randperm(K).int()
        assert order() is None
    assert order() is None


@pytest.mark.gpu
def test_act_order_model_in_inference_mode(monkeypatch):
    """Permutations worked out in inference mode: the same logits as without it, where producers write in the sorted order."""
    monkeypatch.setattr(G, "make_fused_mlp", lambda model: None)
    models = [random_quant_model(hidden=1024, inter=2816, heads=8, layers=2, groupsize=128, seed=83, act_order=True) for _ in range(2)]
    ids = torch.randint(0, 256, (2, 9), device="cuda")

    def logits(model):
        prompt, past = model(ids, use_cache=True)
        step, _ = model(ids[:, :1], past_key_values=past, use_cache=True)
        return prompt, step

    with torch.inference_mode():
        got = logits(models[0])
    with torch.no_grad():
        want = logits(models[1])
    for g, w in zip(got, want):
        assert (g - w).norm() <= 5e-3 * w.norm()  # (the same sums in fp32; fp16 roundings of two layers between them)


@pytest.mark.gpu
def test_first_call_of_an_act_order_block_inside_a_capture(monkeypatch):
    """Nothing is compared (a synchronisation) and nothing kept while a call is being captured: the block gathers for itself there."""
    monkeypatch.setattr(G, "make_fused_mlp", lambda model: None)
    model = random_quant_model(hidden=1024, inter=2816, heads=8, layers=1, groupsize=128, seed=81, act_order=True)
    G.set_layout(model, "stream")
    layer = model.model.layers[0]
    x = torch.randn((2, 1, 1024), device="cuda").half()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    other = random_quant_model(hidden=1024, inter=2816, heads=8, layers=1, groupsize=128, seed=82, act_order=True)
    G.set_layout(other, "stream")
    with torch.cuda.stream(side):                 # workspaces of this stream, from a model of its own
        other.model.layers[0].mlp(x), layer.self_attn.project_qkv(x, torch.zeros((2, 1), dtype=torch.int32, device="cuda"))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out, att = layer.mlp(x), layer.self_attn(hidden_states=x)[0]
    want, want_att = layer.mlp(x), layer.self_attn(hidden_states=x)[0]
    for _ in range(2):
        graph.replay()
        torch.cuda.synchronize()
        assert (out - want).norm() <= 2e-3 * want.norm()   # (separate launches for gate and up: SiLU and product on rounded values)
        assert torch.equal(att, want_att)
        assert torch.equal(layer.mlp(x), want)


@pytest.mark.gpu
@pytest.mark.parametrize("which", ["context", "input"])
def test_another_stream_may_ask_next(which):
    """The stream that works an inverse out is busy: the next call, on another one, is given what is filled already."""
    attn, ways = attention()
    q, order = ways[which]
    q._compact_perm = torch.randperm(K, device="cuda").int()
    torch.cuda.synchronize()
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(first):
        torch.cuda._sleep(10_000_000)
        order()
    with torch.cuda.stream(second):
        got = order().clone()
    torch.cuda.synchronize()
    assert torch.equal(got, inverse_permutation(q._compact_perm))
