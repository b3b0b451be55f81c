"""One token behind a (key, value) pair: every past the block took when it copied it into the new pair."""
import pytest
import torch

import gptq_triton_amd as G
from test_gpu_stream import random_quant_model

pytestmark = pytest.mark.gpu
HEADS, PAST = 8, 37


def strided(t):
    return t.transpose(1, 2).contiguous().transpose(1, 2)


def misaligned(t):
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:]
    return flat.copy_(t.flatten()).view(t.shape)


def halves_of_a_longer_one(t):
    return torch.cat([t, t], dim=2)[:, :, :t.shape[2]]


FORMS = {"float32": lambda t: t.float(), "bfloat16": lambda t: t.bfloat16(), "host": lambda t: t.cpu(), "host float32": lambda t: t.cpu().float(),
         "one for all": lambda t: t[:1], "expanded": lambda t: t[:1].expand(t.shape), "no batch": lambda t: t[0], "strided": strided,
         "misaligned": misaligned, "part": halves_of_a_longer_one}


@pytest.fixture(scope="module")
def model():
    return random_quant_model(hidden=1024, inter=2816, heads=HEADS, layers=2, groupsize=128, seed=61)


def pairs(bsz, past=PAST, layers=2):
    gen = torch.Generator(device="cuda").manual_seed(past)
    # (values that bfloat16 holds as well, the same in every sequence: every form below has the same contents)
    new = lambda: torch.randn((1, HEADS, past, 128), device="cuda", generator=gen).bfloat16().half().expand(bsz, -1, -1, -1).contiguous()
    return [(new(), new()) for _ in range(layers)]


class KeptPair:
    """A transformers Cache of one layer, as far as the attention block asks."""

    def __init__(self, k, v, form=lambda t: t):
        self.k, self.v, self.form = k, v, form

    def get_seq_length(self, layer):
        return self.k.shape[2]

    def update(self, k, v, layer):
        self.k, self.v = (self.form(torch.cat([a, b], dim=2)) for a, b in ((self.k, k), (self.v, v)))
        return self.k, self.v


@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("bsz", [1, 2])
def test_forms_of_the_past(model, form, bsz):
    attn = model.model.layers[0].self_attn
    x = torch.randn((bsz, 1, 1024), device="cuda", generator=torch.Generator(device="cuda").manual_seed(5)).half()
    past = pairs(bsz)
    as_form = [tuple(FORMS[form](t) for t in p) for p in past]
    want, _, (wk, wv) = attn(hidden_states=x, past_key_value=past[0], use_cache=True)
    got, _, (gk, gv) = attn(hidden_states=x, past_key_value=as_form[0], use_cache=True)
    assert torch.equal(got, want) and torch.equal(gk, wk) and torch.equal(gv, wv)
    assert torch.equal(gk[:, :, :PAST], past[0][0]) and torch.equal(gv[:, :, :PAST], past[0][1])
    if form != "no batch":   # (the model reads the length of its past from the third dimension)
        ids = torch.arange(bsz, device="cuda").view(bsz, 1)
        want, new = model(ids, past_key_values=past, use_cache=True)
        got, got_new = model(ids, past_key_values=as_form, use_cache=True)
        assert torch.equal(got, want)
        for a, b in zip(new, got_new):
            assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


def test_a_past_that_takes_a_gradient_stays_in_its_graph(model):
    attn = model.model.layers[0].self_attn
    x = torch.randn((1, 1, 1024), device="cuda").half()
    k, v = (t.requires_grad_() for t in pairs(1)[0])
    _, _, (pk, pv) = attn(hidden_states=x, past_key_value=(k, v), use_cache=True)
    pk.sum().backward()
    assert torch.equal(k.grad, torch.ones_like(k))


def test_an_empty_past_is_no_past(model):
    attn = model.model.layers[0].self_attn
    x = torch.randn((1, 1, 1024), device="cuda").half()
    empty = tuple(torch.empty((1, HEADS, 0, 128), dtype=torch.float16, device="cuda") for _ in range(2))
    want = attn(hidden_states=x)[0]
    assert torch.equal(attn(hidden_states=x, past_key_value=empty)[0], want)


def test_nothing_is_kept_without_use_cache(model):
    """The pairs of all layers are not alive together when the caller does not ask for them."""
    ids = torch.zeros((1, 1), dtype=torch.long, device="cuda")
    past = pairs(1, past=4000)
    model(ids, past_key_values=past), model(ids, past_key_values=past, use_cache=True)   # (tables and workspaces exist)

    def peak(use_cache):
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        out = model(ids, past_key_values=past, use_cache=use_cache)
        del out
        return torch.cuda.max_memory_allocated() - before

    one_layer = 2 * HEADS * 4001 * 128 * 2
    assert peak(False) + one_layer // 2 < peak(True)


@pytest.mark.parametrize("bsz", [1, 2])
@pytest.mark.parametrize("form", ["misaligned", "strided", "part", "one for all", "one head for all"])
def test_forms_of_a_cache(model, form, bsz, monkeypatch):
    """One token with a Cache that hands back its rows in other forms than a contiguous aligned tensor (those may take torch's
    attention, which rounds the probabilities to fp16: 2^-11 of a value each, and the result once more)."""
    attn = model.model.layers[0].self_attn
    monkeypatch.setattr(attn, "layer_idx", 0)
    x = torch.randn((bsz, 1, 1024), device="cuda", generator=torch.Generator(device="cuda").manual_seed(6)).half()
    ids = torch.full((bsz, 1), PAST, dtype=torch.long, device="cuda")
    step = lambda cache: attn(hidden_states=x, position_ids=ids, past_key_values=cache, position_embeddings=())[0]
    part = FORMS.get(form, lambda t: t[:, :1])
    whole = lambda t: part(t).expand(t.shape).clone(memory_format=torch.contiguous_format)
    want, got = step(KeptPair(*pairs(bsz)[0], form=whole)), step(KeptPair(*pairs(bsz)[0], form=part))
    assert (got - want).float().norm() <= 2 ** -9 * want.float().norm()


def test_a_cache_that_takes_a_gradient_stays_in_its_graph(model, monkeypatch):
    attn = model.model.layers[0].self_attn
    monkeypatch.setattr(attn, "layer_idx", 0)
    x = torch.randn((1, 1, 1024), device="cuda").half()
    k, v = (t.requires_grad_() for t in pairs(1)[0])
    seen = []
    hook = attn.o_proj.register_forward_pre_hook(lambda m, args: seen.append(args[0]))
    attn(hidden_states=x, position_ids=torch.full((1, 1), PAST, device="cuda"), past_key_values=KeptPair(k, v), position_embeddings=())
    hook.remove()
    assert seen[0].requires_grad


def test_embedding_rows_with_a_stride(model):
    ids = torch.full((1, 1), 11, dtype=torch.long, device="cuda")
    want = model(ids, past_key_values=pairs(1))[0]
    hook = model.model.embed_tokens.register_forward_hook(lambda m, args, rows: torch.stack([rows, rows], -1)[..., 0])
    try:
        got = model(ids, past_key_values=pairs(1))[0]
    finally:
        hook.remove()
    assert torch.equal(got, want)


def tokens_of(model, bsz):
    dec = G.GreedyDecoder(model, bsz, 32, layout="keep")
    return torch.cat([dec.prefill(torch.arange(3 * bsz, device="cuda").view(bsz, 3)), dec.decode(4)], dim=1)


@pytest.mark.parametrize("layout", ["stream", "checkpoint"])
@pytest.mark.parametrize("bsz", [1, 2, 4, 5])
def test_a_decoder_of_embedding_rows_with_a_stride(model, bsz, layout):
    G.set_layout(model, layout)
    want = tokens_of(model, bsz)
    hook = model.model.embed_tokens.register_forward_hook(lambda m, args, rows: torch.stack([rows, rows], -1)[..., 0])
    try:
        got = tokens_of(model, bsz)
    finally:
        hook.remove()
        G.set_layout(model, "checkpoint")
    assert torch.equal(got, want)


@pytest.mark.parametrize("where", ["input_layernorm", "post_attention_layernorm", "norm"])
@pytest.mark.parametrize("bsz", [1, 2, 4, 5])
def test_norm_weights_with_a_stride(model, bsz, where):
    """Through forward() and through the greedy decoder, in streaming order."""
    G.set_layout(model, "stream")
    norm = model.model.norm if where == "norm" else getattr(model.model.layers[1], where)
    plain = norm.weight
    ids = torch.arange(bsz, device="cuda").view(bsz, 1)
    weights = 1 + 0.1 * torch.randn(1024, device="cuda", generator=torch.Generator(device="cuda").manual_seed(3)).half()
    try:
        norm.weight = torch.nn.Parameter(weights, requires_grad=False)
        want = model(ids, past_key_values=pairs(bsz))[0], tokens_of(model, bsz)
        norm.weight = torch.nn.Parameter(torch.stack([weights, weights], -1)[:, 0], requires_grad=False)
        assert not norm.weight.is_contiguous()
        got = model(ids, past_key_values=pairs(bsz))[0], tokens_of(model, bsz)
    finally:
        norm.weight = plain
        G.set_layout(model, "checkpoint")
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
