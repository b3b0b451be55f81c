"""GreedyDecoder goes on from its state buffers whoever moved them: decode() after a step that was interrupted on the host, after the
caller replayed the captured graph, and after the caller wrote to the position or the tokens."""
import pytest
import torch

import gptq_triton_amd as G
from gptq_triton_amd.fused_attention import LlamaConfigLite
from gptq_triton_amd.llama import GreedyDecoder, LlamaForCausalLM
from test_loader import make_checkpoint

CAPACITY = 20


def token_at(place, b):
    return 7 * place + 3 * b + 1


class Interrupted(Exception):
    pass


def decoder_of_known_tokens(monkeypatch, bsz=2):
    """A decoder on the CPU whose step does to the state buffers what the launch at the end of a step does: moves them on through
    raw memory, without a trace in the tensors' version counters.  The token at place p of sequence b is token_at(p, b)."""
    cfg = LlamaConfigLite(hidden_size=64, num_attention_heads=2, intermediate_size=64, num_hidden_layers=1, vocab_size=512)
    monkeypatch.setattr(GreedyDecoder, "one_launch_end", True, raising=False)
    dec = GreedyDecoder(LlamaForCausalLM(cfg), bsz, CAPACITY)
    vars(dec).pop("one_launch_end", None)
    dec.fail_in = None  # steps until one is interrupted

    def step():
        if dec.fail_in is not None:
            if dec.fail_in == 0:
                dec.fail_in = None
                raise Interrupted
            dec.fail_in -= 1
        dec.position.data.add_(1)
        for b in range(bsz):
            at = int(dec.position[b, 0])
            dec.tokens.data[b, 0] = token_at(at, b)
            if 0 <= at <= CAPACITY:
                dec.history.data[b, at] = token_at(at, b)

    monkeypatch.setattr(dec, "_step", step)
    monkeypatch.setattr(dec, "_layers", lambda *a, **k: torch.tensor([[token_at(5, b)] for b in range(bsz)]))
    dec.prefill(torch.zeros((bsz, 5), dtype=torch.long))
    return dec


def want(first, steps, bsz=2):
    return torch.tensor([[token_at(first + i, b) for i in range(steps)] for b in range(bsz)])


@pytest.mark.parametrize("moved", ["interrupted", "stepped", "data", "replaced"])
def test_decode_goes_on_from_where_the_kernels_left_the_sequences(monkeypatch, moved):
    dec = decoder_of_known_tokens(monkeypatch)
    assert torch.equal(dec.decode(2), want(6, 2))       # places 6, 7
    if moved == "interrupted":
        dec.fail_in = 2
        with pytest.raises(Interrupted):
            dec.decode(4)
    elif moved == "stepped":                            # (as a replay of the captured graph by the caller)
        dec._step()
        dec._step()
    elif moved == "data":
        dec.position.data.fill_(9)
    else:
        dec.position = torch.full_like(dec.position, 9)
    assert torch.equal(dec.decode(3), want(10, 3))      # standing at 9
    with pytest.raises(ValueError):
        dec.decode(CAPACITY - 12 + 1)                   # standing at 12
    assert torch.equal(dec.decode(CAPACITY - 12), want(13, CAPACITY - 12))


def test_decode_of_no_and_of_fewer_steps(monkeypatch):
    dec = decoder_of_known_tokens(monkeypatch)
    assert dec.decode(0).shape == (2, 0)
    with pytest.raises(RuntimeError):
        dec.decode(-1)
    assert torch.equal(dec.decode(2), want(6, 2))


def test_decode_of_sequences_at_different_places(monkeypatch):
    dec = decoder_of_known_tokens(monkeypatch)
    dec.position.copy_(torch.tensor([[4], [9]]))
    got = dec.decode(3)
    assert got.tolist() == [[token_at(5 + i, 0) for i in range(3)], [token_at(10 + i, 1) for i in range(3)]]
    with pytest.raises(ValueError):
        dec.decode(CAPACITY - 12 + 1)


def test_a_step_starts_from_the_tokens_buffer(monkeypatch):
    monkeypatch.setattr(GreedyDecoder, "one_launch_end", True, raising=False)
    cfg = LlamaConfigLite(hidden_size=64, num_attention_heads=2, intermediate_size=64, num_hidden_layers=1, vocab_size=512)
    model = LlamaForCausalLM(cfg)
    dec = GreedyDecoder(model, 2, CAPACITY)
    if not dec.one_launch_end:
        dec.one_launch_end = True
    seen = []
    monkeypatch.setattr(dec, "_layers", lambda h, *a, **k: seen.append(h.clone()))
    dec.tokens.copy_(torch.tensor([[17], [400]]))
    dec._step()
    assert torch.equal(seen[0], model.model.embed_tokens(dec.tokens))


def test_an_lm_head_replaced_later(monkeypatch):
    """The one-launch end is chosen by the lm_head there is at the step, not by the one the decoder was made with."""
    from gptq_triton_amd import llama
    cfg = LlamaConfigLite(hidden_size=64, num_attention_heads=2, intermediate_size=64, num_hidden_layers=1, vocab_size=512)
    model = LlamaForCausalLM(cfg)
    launches = []
    monkeypatch.setattr(llama, "head_argmax_takes", lambda rows, weight: weight.shape[0] == 512)
    monkeypatch.setattr(llama, "greedy_step_end", lambda *a: launches.append(a))
    dec = GreedyDecoder(model, 2, CAPACITY)
    x = torch.randn(2, 1, 64)
    dec._end_step(None, None, model.model.norm, x)
    assert len(launches) == 1
    model.lm_head = torch.nn.Linear(64, 300, bias=False)
    dec._end_step(None, None, model.model.norm, x)
    assert len(launches) == 1 and torch.equal(dec.tokens, model.lm_head(x).argmax(-1)) and dec.position.tolist() == [[1], [1]]
    model.lm_head = torch.nn.Linear(64, 512, bias=False)
    dec._end_step(None, None, model.model.norm, x)
    assert len(launches) == 2
    model.lm_head = torch.nn.Embedding(512, 64)         # (tied weights: a module that has no bias at all)
    dec._end_step(None, None, model.model.norm, x)
    assert len(launches) == 3


@pytest.mark.gpu
def test_decoder_whose_lm_head_is_replaced(tmp_path):
    """An lm_head the launch does not take (a strided weight) after a few steps: the decoder goes on, with the same tokens."""
    cfg = make_checkpoint(tmp_path, 128, seed=33)
    model = G.load_quant(str(tmp_path), device="cuda", fuse_mlp=True)
    ids = torch.arange(6, device="cuda").view(1, 6)
    want = model.generate_greedy(ids, 13)[:, 6:]
    dec = GreedyDecoder(model, 1, 24)
    got = [dec.prefill(ids), dec.decode(4)]
    assert dec.one_launch_end
    weight = model.lm_head.weight
    model.lm_head.weight = torch.nn.Parameter(weight.t().contiguous().t(), requires_grad=False)
    assert not dec.one_launch_end
    got += [dec.decode(4), dec.decode(2, use_graph=True)]
    model.lm_head.weight = weight
    got.append(dec.decode(2))
    assert torch.equal(torch.cat(got, dim=1), want)


@pytest.mark.gpu
@pytest.mark.parametrize("bsz", [1, 3])
def test_replays_follow_tokens_and_prompts_written_between_them(tmp_path, bsz):
    """decoder.graph after another prefill, and after the caller put other tokens in place (a sampling loop on the graph)."""
    cfg = make_checkpoint(tmp_path, 128, seed=32)
    model = G.load_quant(str(tmp_path), device="cuda", fuse_mlp=True)
    torch.manual_seed(8)
    ids, other = torch.randint(0, cfg.vocab_size, (2, bsz, 6)).cuda()
    forced = torch.randint(0, cfg.vocab_size, (bsz, 1)).cuda()
    graph, eager = GreedyDecoder(model, bsz, 24), GreedyDecoder(model, bsz, 24)
    graph.prefill(ids)
    graph.decode(3, use_graph=True)
    graph.prefill(other), eager.prefill(other)
    for _ in range(3):
        graph.graph.replay(), eager.decode(1)
        assert torch.equal(graph.tokens, eager.tokens) and torch.equal(graph.position, eager.position)
        graph.tokens.copy_(forced), eager.tokens.copy_(forced)
    assert torch.equal(graph.decode(2, use_graph=True), eager.decode(2))


@pytest.mark.gpu
@pytest.mark.parametrize("use_graph", [False, True])
@pytest.mark.parametrize("bsz", [1, 3])
def test_decode_after_an_interrupted_and_an_outside_step(tmp_path, monkeypatch, bsz, use_graph):
    cfg = make_checkpoint(tmp_path, 128, seed=31)
    model = G.load_quant(str(tmp_path), device="cuda", fuse_mlp=True)
    torch.manual_seed(7)
    ids = torch.randint(0, cfg.vocab_size, (bsz, 6)).cuda()
    straight = GreedyDecoder(model, bsz, 24)
    tokens = [straight.prefill(ids), straight.decode(16)]
    tokens = torch.cat(tokens, dim=1)                   # 17 tokens, places 6 .. 22

    dec = GreedyDecoder(model, bsz, 24)
    assert torch.equal(dec.prefill(ids), tokens[:, :1])
    assert torch.equal(dec.decode(3, use_graph=use_graph), tokens[:, 1:4])
    real, left = GreedyDecoder._step, [2]

    def interrupted(self):
        if left[0] == 0:
            raise Interrupted
        left[0] -= 1
        real(self)

    with monkeypatch.context() as m:
        m.setattr(GreedyDecoder, "_step", interrupted)
        with pytest.raises(Interrupted):
            dec.decode(5)                               # two of five steps are done
    assert torch.equal(dec.decode(2, use_graph=use_graph), tokens[:, 6:8])
    if use_graph:
        dec.graph.replay()
    else:
        dec._step()
    assert torch.equal(dec.tokens, tokens[:, 8:9])
    assert torch.equal(dec.decode(4, use_graph=use_graph), tokens[:, 9:13])
    with pytest.raises(ValueError):
        dec.decode(7, use_graph=use_graph)              # standing at place 18 of 24
    assert torch.equal(dec.decode(4, use_graph=use_graph), tokens[:, 13:17])
