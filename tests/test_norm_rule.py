"""Which decode steps put the residual add and the RMSNorm into the projection's own launch."""
import pytest
import torch

import gptq_triton_amd as G
from gptq_triton_amd.llama import LlamaMLP
from test_gpu_stream import random_quant_model


def blocks(hidden, inter, act_order):
    """The attention block and both MLP blocks as they stand in streaming order (nothing is launched)."""
    def new(k, n):
        layer = G.QuantLinear(4, 128, k, n, bias=False, act_order=act_order)
        layer._stream_meta, layer._stream_rows = torch.zeros(1, dtype=torch.int32), 16
        layer._compact_perm = torch.arange(k, dtype=torch.int32) if act_order else None
        return layer

    cfg = G.LlamaConfigLite()
    cfg.hidden_size, cfg.intermediate_size, cfg.num_attention_heads = hidden, inter, hidden // 128
    with torch.device("meta"):
        attn = G.QuantLlamaAttention(cfg, new(hidden, 3 * hidden), new(hidden, hidden))
        mlp = LlamaMLP(cfg)
        mlp.gate_proj, mlp.up_proj, mlp.down_proj = new(hidden, inter), new(hidden, inter), new(inter, hidden)
        plain = [G.QuantLinear(4, 128, k, n, bias=False, act_order=False) for k, n in ((hidden, inter), (inter, hidden), (hidden, inter))]
        fused = G.QuantLlamaMLP(*plain)
    fused._gate_meta, fused._stream_rows = torch.zeros(1, dtype=torch.int32), 16
    if act_order:
        order = torch.arange(hidden, dtype=torch.int32)
        fused.g_idx = fused._compact_rows = mlp.gate_proj._compact_perm = mlp.up_proj._compact_perm = order
    return attn, mlp, fused


@pytest.mark.parametrize("act_order", [False, True])
@pytest.mark.parametrize("hidden,inter", [(1024, 2816), (4096, 11008), (4352, 11776), (6656, 17920), (8192, 22016)])
def test_rows_that_take_the_norm_along(hidden, inter, act_order):
    """Up to four; three with act-order and rows that every workgroup would gather for longer than a norm launch takes."""
    most = 3 if act_order and hidden > 4096 else 4
    for block in blocks(hidden, inter, act_order):
        assert [block.norm_fusable(rows) for rows in range(6)] == [0 < rows <= most for rows in range(6)], type(block)


def test_rows_follow_the_tuning_of_the_launches():
    """The rows a launch normalises are asked for under the launch shape of the moment: sixteen waves with two matrices leave less
    room for the rows."""
    from gptq_triton_amd import _lib
    from gptq_triton_amd.quant_linear import stream_norm_rows
    shapes = [(op, k, n) for k in (1024, 4096, 6656, 8192) for op, n in ((_lib.OP_QKV_ROTARY, 3 * k), (_lib.OP_MLP_GATEUP, 4096))]
    ask = lambda: [stream_norm_rows(op, k, n, 128) for op, k, n in shapes]
    before = ask()
    _lib.load().gptq4_set_stream_tuning(16, 1)
    fresh = [_lib.load().gptq4_stream_rows(op | _lib.OP_WITH_NORM, k, n, 128) for op, k, n in shapes]
    assert ask() == fresh != before
    _lib.load().gptq4_set_stream_tuning(0, 0)
    assert ask() == before


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["stream", "checkpoint"])
@pytest.mark.parametrize("act_order", [False, True])
@pytest.mark.parametrize("fuse_mlp", [False, True])
@pytest.mark.parametrize("bsz", [1, 2, 4, 5])
def test_steps_take_the_norm_along_by_default(monkeypatch, bsz, fuse_mlp, act_order, layout):
    """Decode steps and forward() of up to four sequences in streaming order, of one in checkpoint order where gate and up are
    fused (unfused they are launches of their own there): tokens, logits and pairs are those of the layer with norm launches."""
    from gptq_triton_amd import decoder_ops
    if not fuse_mlp:
        monkeypatch.setattr(G, "make_fused_mlp", lambda model: None)
    model = random_quant_model(hidden=1024, inter=2816, heads=8, layers=2, groupsize=128, seed=71, act_order=act_order)
    G.set_layout(model, layout)
    ids = torch.randint(0, model.config.vocab_size, (bsz, 9), device="cuda", generator=torch.Generator(device="cuda").manual_seed(bsz))
    _, past = model(ids[:, :8], use_cache=True)
    taken = []
    for block in {type(layer.mlp) for layer in model.model.layers}:
        real = block.forward_normed
        monkeypatch.setattr(block, "forward_normed", lambda self, *a, real=real: taken.append(1) or real(self, *a))

    def step():
        dec = G.GreedyDecoder(model, bsz, 32, layout="keep")
        tokens = [dec.prefill(ids)]
        del taken[:]
        tokens.append(dec.decode(4))
        decoded = len(taken)
        del taken[:]
        logits, pairs = model(ids[:, 8:], past_key_values=past, use_cache=True)
        return decoded, len(taken), tokens + [logits] + [t for pair in pairs for t in pair]

    inside = bsz <= 4 if layout == "stream" else bsz == 1 and fuse_mlp
    decoded, forward, got = step()
    assert (decoded, forward) == ((8, 2) if inside else (0, 0))
    with monkeypatch.context() as mp:
        mp.setattr(decoder_ops, "NORM_PAYS_ROWS", 0)
        decoded, forward, want = step()
    assert decoded == forward == 0 and all(torch.equal(a, b) for a, b in zip(got, want))
