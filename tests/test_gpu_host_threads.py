"""The extension behind the operators from several threads and streams: calls give up the interpreter lock around a launch, and every
stream has a workspace of its own that grows on its first larger call."""
import threading

import pytest
import torch

import gptq_triton_amd as G
from gptq_triton_amd import _lib, decoder_ops, quant_linear as Q
from test_gpu_stream import random_quant_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("own_streams", [True, False])
def test_operators_from_several_threads(own_streams):
    """Projections that exchange partial sums through the workspace, norms, the MLP and one-token attention, from four threads:
    every result is that of the same call alone."""
    model = random_quant_model(hidden=1024, inter=2816, heads=8, layers=2, groupsize=128, seed=91)
    G.set_layout(model, "stream")
    layer = model.model.layers[0]
    gen = torch.Generator(device="cuda").manual_seed(4)
    new = lambda *s: torch.randn(s, device="cuda", generator=gen).half()
    weight = new(1024)

    def work(t):
        past = tuple(new(1, 8, 30 + t, 128) for _ in range(2))
        jobs = []
        for rows in (1, 3, 9, 40, 200 + 64 * t, 1000 + 500 * t):    # (the last ones make the workspaces grow)
            x = new(1, rows, 1024)
            jobs += [lambda x=x: layer.mlp(x), lambda x=x: layer.self_attn.o_proj(x), lambda x=x: decoder_ops.rms_norm(x, weight, 1e-6)]
        one = new(1, 1, 1024)
        jobs.append(lambda: layer.self_attn(hidden_states=one, past_key_value=past)[0])
        return jobs

    jobs = [work(t) for t in range(4)]
    want = [[job().clone() for job in todo] for todo in jobs]
    torch.cuda.synchronize()
    failed, start = [], threading.Barrier(4)

    def run(t):
        try:
            stream = torch.cuda.Stream() if own_streams else torch.cuda.current_stream()
            with torch.cuda.stream(stream):
                start.wait()
                for turn in range(5):
                    got = [job() for job in jobs[t]]
                    stream.synchronize()
                    for i, (a, b) in enumerate(zip(got, want[t])):
                        if not torch.equal(a, b):
                            failed.append((t, turn, i))
        except Exception as e:  # noqa: BLE001 - reported by the test's own thread
            failed.append((t, repr(e)))

    threads = [threading.Thread(target=run, args=(t,)) for t in range(4)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not failed, failed
    assert _lib.exchange_errors() == []


def test_a_workspace_that_grows_while_its_stream_is_busy():
    """Calls of growing size on one stream without a wait in between: the outgrown workspaces stay alive under their launches."""
    k, n, g = 2048, 1024, 128
    gen = torch.Generator(device="cuda").manual_seed(6)
    w = torch.randint(-2 ** 31, 2 ** 31 - 1, (k // 8, n), dtype=torch.int32, device="cuda", generator=gen)
    z = torch.randint(-2 ** 31, 2 ** 31 - 1, (k // g, n // 8), dtype=torch.int32, device="cuda", generator=gen)
    s = (0.01 * torch.rand((k // g, n), device="cuda", generator=gen)).half()
    xs = [torch.randn((m, k), device="cuda", generator=gen).half() for m in (1, 5, 17, 64, 300, 2000)]
    want = [Q.matmul4(g, x, w, s, z) for x in xs]
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.Stream()) as _:
        got = [Q.matmul4(g, x, w, s, z) for x in xs for _ in range(3)]
        torch.cuda.current_stream().synchronize()
    for i, y in enumerate(got):
        assert torch.equal(y, want[i // 3])
