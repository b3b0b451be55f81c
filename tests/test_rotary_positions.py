"""The positions a caller of the attention block does not pass: kept per stream, never inside a captured graph."""
import pytest
import torch

import gptq_triton_amd as G
from gptq_triton_amd import _lib
from test_loader import make_checkpoint


@pytest.fixture
def on_cpu(monkeypatch):
    """RotaryTable.positions on the CPU, with the stream and its capture state to choose."""
    state = {"stream": 0, "capturing": False}
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: state["capturing"])
    monkeypatch.setattr(_lib, "current_stream", lambda device: state["stream"])
    return state


CPU = torch.device("cpu", 0)


def test_positions_of_one_stream_are_not_read_on_another(on_cpu):
    rope = G.RotaryTable(128, 32)
    first = rope.positions(CPU, 3, 2, 1)
    assert first.tolist() == [[3], [3]] and rope.positions(CPU, 3, 2, 1).data_ptr() == first.data_ptr()
    on_cpu["stream"] = 1
    assert rope.positions(CPU, 3, 2, 1).data_ptr() != first.data_ptr()


def test_a_captured_call_neither_reads_nor_leaves_a_table(on_cpu):
    rope = G.RotaryTable(128, 32)
    kept = rope.positions(CPU, 3, 2, 1)
    on_cpu["capturing"] = True
    assert rope.positions(CPU, 3, 2, 1).data_ptr() != kept.data_ptr()
    mine = rope.positions(CPU, 5, 4, 1)
    assert mine.tolist() == [[5]] * 4 and rope.positions(CPU, 5, 1, 3).tolist() == [[5, 6, 7]]
    on_cpu["capturing"] = False
    mine.fill_(-1)                       # (the graph's own memory)
    assert rope.positions(CPU, 5, 4, 1).tolist() == [[5]] * 4


def test_positions_past_the_table_are_not_a_table_each(on_cpu, monkeypatch):
    rope = G.RotaryTable(128, 32)
    made = []
    real = torch.arange
    monkeypatch.setattr(torch, "arange", lambda *a, **k: made.append(a) or real(*a, **k))
    for start in range(30, 230):
        assert rope.positions(CPU, start, 1, 1).tolist() == [[start]]
    assert len(made) <= 4, made
    for bsz in range(2, 40):             # bounded, and right, for any number of batch sizes
        assert rope.positions(CPU, 7, bsz, 1).tolist() == [[7]] * bsz
    assert len(rope._counts) <= 16


@pytest.mark.gpu
def test_graph_over_the_attention_block_keeps_its_positions(tmp_path):
    """A graph captured over one-token attention, replayed after the block has served many other batch sizes and streams; and
    eager calls of a batch size that was first seen in a capture."""
    make_checkpoint(tmp_path, 128, seed=41)
    model = G.load_quant(str(tmp_path), device="cuda", fuse_mlp=True)
    attn = model.model.layers[0].self_attn
    gen = torch.Generator(device="cuda").manual_seed(3)

    def inputs(bsz, past=9):
        new = lambda *s: torch.randn(s, device="cuda", generator=gen).half()
        return new(bsz, 1, 256), (new(bsz, 2, past, 128), new(bsz, 2, past, 128))

    def run(x, past):
        return attn(hidden_states=x, past_key_value=past, use_cache=True)

    x, past = inputs(3)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):        # everything but the positions of three sequences exists on this stream
        run(*inputs(2))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out, _, pair = run(x, past)
    want, _, want_pair = run(x, past)    # eager, before the first replay
    for _ in range(2):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(pair[0], want_pair[0]) and torch.equal(pair[1], want_pair[1])
        for bsz in range(4, 24):         # more batch sizes than tables are kept for, and other contents in what was freed
            run(*inputs(bsz))
        torch.cuda.empty_cache()
        junk = [torch.full((512, b), 400, dtype=torch.int32, device="cuda") for b in range(1, 24)]
        with torch.cuda.stream(side):
            side.wait_stream(torch.cuda.current_stream())
            again, _, _ = run(x, past)
        torch.cuda.synchronize()
        assert torch.equal(again, want)
        del junk
