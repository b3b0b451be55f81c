"""gptq4_lm_head_argmax (decoder_ops.lm_head_argmax): the fp16 lm_head GEMV and the greedy argmax in one launch.
The logits are fp32 sums rounded to fp16 once; a library GEMV may round differently by an ulp, so on random data the
chosen index is checked against float64 logits (it must be within two fp16 ulps of the true maximum), and exactly on
data with a planted winner and on exact ties (the lower index wins, as torch.argmax)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def ops():
    from gptq_triton_amd import decoder_ops
    return decoder_ops


def head_is_zero():
    from gptq_triton_amd import _lib
    torch.cuda.synchronize()
    return all(int(ws[:_lib.WS_HEAD_BYTES].view(torch.int64).abs().sum()) == 0 for ws in _lib._workspaces.values())


@pytest.mark.parametrize("b,k,v", [(1, 4096, 32000), (8, 5120, 32000), (16, 4096, 32001), (3, 6656, 1000), (2, 8192, 5003), (1, 4096, 17)])
def test_against_float64_logits(b, k, v):
    rng = np.random.default_rng(b + k + v)
    x = rng.standard_normal((b, k)).astype(np.float16)
    w = (0.02 * rng.standard_normal((v, k))).astype(np.float16)
    out = ops().lm_head_argmax(torch.from_numpy(x).cuda().view(b, 1, k), torch.from_numpy(w).cuda(), max_rows=16)
    assert out.shape == (b, 1) and out.dtype == torch.int64
    logits = x.astype(np.float64) @ w.astype(np.float64).T
    got = out.cpu().numpy().reshape(b)
    for i in range(b):
        top = logits[i].max()
        assert 0 <= got[i] < v
        assert logits[i, got[i]] >= top - 2 * float(np.spacing(np.float16(abs(top)))), (i, got[i], int(logits[i].argmax()))
    assert head_is_zero()


def test_planted_winner_and_ties():
    rng = np.random.default_rng(5)
    b, k, v = 4, 4096, 32000
    x = rng.standard_normal((b, k)).astype(np.float16)
    w = (0.01 * rng.standard_normal((v, k))).astype(np.float16)
    winners = [31999, 0, 12345, 20000]
    for i, r in enumerate(winners):
        w[r] = (x[i].astype(np.float32) * 0.05).astype(np.float16)   # logit ~ 0.05 * |x|^2 = 200, far above the rest
    w[100] = w[20000]   # an exact tie for row 3: the lower index wins
    xd, wd = torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda()
    out = ops().lm_head_argmax(xd, wd)
    assert out.tolist() == [31999, 0, 12345, 100]
    assert torch.equal(out, torch.nn.functional.linear(xd, wd).argmax(-1))
    # the same twice: nothing is left behind in the workspace
    assert torch.equal(ops().lm_head_argmax(xd, wd), out) and head_is_zero()


def test_other_shapes_go_through_torch():
    x = torch.randn(2, 1000, device="cuda").half()
    w = torch.randn(50, 1000, device="cuda").half()
    assert torch.equal(ops().lm_head_argmax(x, w), torch.nn.functional.linear(x, w).argmax(-1))
    from gptq_triton_amd import _lib
    lib = _lib.load()
    fake = 0x1000
    assert lib.gptq4_lm_head_argmax(fake, fake, fake, 1, 4000, 32000, fake, _lib.WS_HEAD_BYTES + (64 << 10), None) == -2
    assert lib.gptq4_lm_head_argmax(fake, fake, fake, 17, 4096, 32000, fake, _lib.WS_HEAD_BYTES + (64 << 10), None) == -2
    assert lib.gptq4_lm_head_argmax(fake, fake, fake, 1, 4096, 32000, fake, 64, None) == -4
    assert lib.gptq4_lm_head_argmax(None, fake, fake, 1, 4096, 32000, fake, _lib.WS_HEAD_BYTES + (64 << 10), None) == -1


@pytest.mark.parametrize("b,k,v", [(1, 256, 16), (5, 1280, 333), (1, 7680, 2001), (16, 4864, 257), (9, 2048, 50257)])
def test_any_multiple_of_256(b, k, v):
    """Row lengths and vocabularies of no particular size, against torch on the same tensors: logits are fp32 sums rounded to
    fp16 on both sides, so the chosen logit is within two fp16 ulps of the largest."""
    gen = torch.Generator(device="cuda").manual_seed(b * k + v)
    x = torch.randn((b, k), device="cuda", generator=gen).half()
    w = (0.02 * torch.randn((v, k), device="cuda", generator=gen)).half()
    out = ops().lm_head_argmax(x, w)
    logits = x.double() @ w.double().t()
    top = logits.max(1).values
    got = logits.gather(1, out[:, None])[:, 0]
    assert ((top - got) <= 2 * 2.0 ** -10 * top.abs()).all(), (top - got).max()
    assert head_is_zero()


@pytest.mark.parametrize("b,k,norm", [(1, 1024, "add"), (1, 8192, "plain"), (1, 1280, None), (6, 4096, None)])
def test_step_end_moves_the_loop_on(b, k, norm):
    """One launch = the norm launch, the argmax launch and the bookkeeping of a greedy loop, bit for bit."""
    gen = torch.Generator(device="cuda").manual_seed(k + b)
    new = lambda *s: torch.randn(s, device="cuda", generator=gen).half()
    v, cap = 1003, 9
    x, delta, nw = new(b, 1, k), new(b, 1, k), (1 + 0.1 * new(k)).half()
    w, embed = (0.02 * new(v, k)).half(), new(v, k)
    tokens = torch.zeros((b, 1), dtype=torch.int64, device="cuda")
    pos = torch.arange(b, dtype=torch.int32, device="cuda")[:, None].contiguous() + 3
    history = torch.full((b, cap), -1, dtype=torch.int64, device="cuda")
    hidden = torch.zeros((b, 1, k), dtype=torch.float16, device="cuda")
    normed = x if norm is None else ops().add_rms_norm(x, delta, nw, 1e-6)[1] if norm == "add" else ops().rms_norm(x, nw, 1e-6)
    want = ops().lm_head_argmax(normed, w)
    ops().greedy_step_end(x, delta if norm == "add" else None, None if norm is None else nw, 1e-6, w, tokens, pos, history, embed, hidden)
    assert torch.equal(tokens, want)
    assert pos[:, 0].tolist() == [4 + i for i in range(b)]
    assert torch.equal(hidden[:, 0], embed[want[:, 0]])
    expect = torch.full_like(history, -1)
    for i in range(b):
        if 4 + i < cap:   # (a place past the end is not written)
            expect[i, 4 + i] = want[i, 0]
    assert torch.equal(history, expect) and head_is_zero()


@pytest.mark.parametrize("b,k,v", [(1, 4096, 32000), (3, 1024, 700), (16, 512, 1003)])
def test_nan_and_infinite_logits(b, k, v):
    """NaN counts as the largest logit, infinities as numbers, the lowest index among equals: torch.argmax of the same logits."""
    gen = torch.Generator(device="cuda").manual_seed(b + k)
    x = (0.5 + torch.rand((b, k), device="cuda", generator=gen)).half()   # positive: a row of one sign has a logit of that sign
    w = (0.02 * torch.randn((v, k), device="cuda", generator=gen)).half()
    nan, inf = float("nan"), float("inf")

    def check(expect, x=x):
        assert ops().lm_head_argmax(x, w).tolist() == expect
        tokens = torch.zeros((b, 1), dtype=torch.int64, device="cuda")
        pos = torch.zeros((b, 1), dtype=torch.int32, device="cuda")
        ops().greedy_step_end(x.view(b, 1, k), None, None, 1e-6, w, tokens, pos, torch.zeros((b, 4), dtype=torch.int64, device="cuda"))
        assert tokens[:, 0].tolist() == expect
        assert torch.nn.functional.linear(x, w).argmax(-1).tolist() == expect

    w[v - 3, k // 2] = inf
    check([v - 3] * b)
    w[5, 1] = inf
    check([5] * b)
    w[v // 2, 7] = nan
    check([v // 2] * b)
    w[v - 1, 0] = nan
    check([v // 2] * b)
    w[2, k - 1] = nan
    check([2] * b)
    bad = x.clone()
    bad[b - 1, 3] = nan        # every logit of the last row
    check([2] * (b - 1) + [0], bad)
    w.fill_(-inf)
    check([0] * b)
    assert head_is_zero()


@pytest.mark.parametrize("b", [1, 4, 6, 16])
def test_equal_logits_side_by_side(b):
    """The lowest index among equal logits and NaN wherever the equals lie: next to each other (rows of one product, which
    different lanes compare), one wave or one workgroup apart."""
    k, v = 512, 8192   # 32 rows a workgroup of 256, four a wave
    gen = torch.Generator(device="cuda").manual_seed(b)
    x = (0.5 + torch.rand((b, k), device="cuda", generator=gen)).half()
    for first in (0, 1, 2, 3, 30, 4097):
        for step in (1, 2, 3, 4, 32):
            for value in (0.5, float("nan")):
                w = (0.001 * torch.randn((v, k), device="cuda", generator=gen)).half()
                w[first::step][:5] = value
                assert ops().lm_head_argmax(x, w).tolist() == [first] * b, (first, step, value)
    assert ops().lm_head_argmax(torch.zeros_like(x), w.nan_to_num()).tolist() == [0] * b   # all of them
    assert head_is_zero()


def off_by_one(t):
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:]
    return flat.copy_(t.flatten()).view(t.shape)


@pytest.mark.parametrize("b", [1, 5, 16])
@pytest.mark.parametrize("which", ["x", "weight", "both"])
def test_operands_off_the_16_byte_grid(b, which):
    """Views into a flat buffer: the library reads 16 bytes at a time and refuses them, the function does not."""
    gen = torch.Generator(device="cuda").manual_seed(b)
    x = torch.randn((b, 1, 2048), device="cuda", generator=gen).half()
    w = 0.02 * torch.randn((1000, 2048), device="cuda", generator=gen).half()
    best = torch.arange(b, device="cuda") * 7 + 3
    w[best] = 0.05 * x[:, 0]   # row `best` wins by far: its logit is about 100 where the others' spread is about 1
    got = ops().lm_head_argmax(off_by_one(x) if which != "weight" else x, off_by_one(w) if which != "x" else w)
    assert torch.equal(got.view(-1), best)


@pytest.mark.parametrize("b", [1, 2, 4, 5, 9, 16])
@pytest.mark.parametrize("k,v", [(256, 1), (768, 3), (1280, 255), (4096, 1031), (4864, 2049)])
def test_logits_against_float64(b, k, v):
    """Rows that do not fill a tile, a wave or a workgroup, and row lengths that end within a group of loads.  Every logit is
    within half an fp16 ulp plus the bound of k fp32 additions in any order of the exact sum."""
    gen = torch.Generator(device="cuda").manual_seed(b + k + v)
    x = torch.randn((b, 1, k), device="cuda", generator=gen).half()
    w = 0.02 * torch.randn((v, k), device="cuda", generator=gen).half()
    y = ops().lm_head_logits(x, w)
    assert y.shape == (b, 1, v) and y.dtype == torch.float16
    xd, wd = x.view(b, k).double().cpu(), w.double().cpu()
    exact, size = xd @ wd.t(), xd.abs() @ wd.abs().t()
    err = (y.view(b, v).double().cpu() - exact).abs()
    assert bool((err <= exact.abs() * 2.0 ** -11 + size * k * 2.0 ** -24 + 2.0 ** -25).all()), float((err / size).max())
    assert torch.equal(ops().lm_head_argmax(x, w).view(b), y.view(b, v).argmax(-1))   # the same sums


@pytest.mark.parametrize("b", [1, 6])
def test_subnormal_weights_count(b):
    """fp16 weights below 2^-14 are values, not zeros, in the matrix products."""
    gen = torch.Generator(device="cuda").manual_seed(b)
    x = 64 * torch.randn((b, 1024), device="cuda", generator=gen).half()
    w = (2.0 ** -17 * torch.randn((77, 1024), device="cuda", generator=gen)).half()
    exact = x.double() @ w.double().t()
    size = x.double().abs() @ w.double().abs().t()
    assert bool(((ops().lm_head_logits(x, w).double() - exact).abs() <= exact.abs() * 2.0 ** -11 + size * 1024 * 2.0 ** -24 + 2.0 ** -25).all())


def test_logits_of_a_weight_that_is_more_than_a_tensor():
    """A weight of a tensor subclass, and a vocabulary of none, take torch's linear layer as before."""
    from gptq_triton_amd.llama import LlamaForCausalLM

    class Counted(torch.Tensor):
        calls = 0

        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            cls.calls += func is torch.nn.functional.linear
            return super().__torch_function__(func, types, args, kwargs or {})

    model = LlamaForCausalLM.__new__(LlamaForCausalLM)
    torch.nn.Module.__init__(model)
    model.lm_head = torch.nn.Linear(512, 300, bias=False).cuda().half()
    h = torch.randn((3, 1, 512), device="cuda").half()
    with torch.no_grad():
        model.lm_head.weight = torch.nn.Parameter(model.lm_head.weight.detach().as_subclass(Counted), requires_grad=False)
        assert model._logits(h).shape == (3, 1, 300) and Counted.calls == 1
        model.lm_head = torch.nn.Linear(512, 300, bias=False).cuda().half()
        model.lm_head.weight = torch.nn.Parameter(torch.empty((0, 512), device="cuda", dtype=torch.float16))
        assert model._logits(h).shape == (3, 1, 0)


def test_logits_of_a_model_with_a_hook_on_its_lm_head():
    """forward() calls an lm_head that a hook hangs on, and gives torch's logits within an fp16 ulp where none does."""
    from gptq_triton_amd.llama import LlamaForCausalLM
    head = torch.nn.Linear(512, 300, bias=False).cuda().half()
    model = LlamaForCausalLM.__new__(LlamaForCausalLM)
    torch.nn.Module.__init__(model)
    model.lm_head = head
    h = torch.randn((3, 1, 512), device="cuda").half()
    with torch.no_grad():
        own, torchs = model._logits(h), head(h)
        assert float((own.float() - torchs.float()).abs().max()) <= 2.0 ** -10 * float(torchs.abs().max())
        calls = []
        handle = head.register_forward_hook(lambda m, i, o: calls.append(1) or o + 1)
        assert torch.equal(model._logits(h), torchs + 1) and calls
        handle.remove()
        head.bias = torch.nn.Parameter(torch.ones(300, device="cuda").half())
        assert torch.equal(model._logits(h), head(h))


class Doubled(torch.nn.Linear):
    def forward(self, x):
        return 2 * super().forward(x)


class Marked(torch.Tensor):
    pass


def hooked(head):
    head.register_forward_hook(lambda m, args, out: out + 1)
    return head


def with_bias(head):
    head.bias = torch.nn.Parameter(torch.ones(8192, device="cuda").half())
    return head


def with_weight(change):
    def made(head):
        head.weight = torch.nn.Parameter(change(head.weight.detach()), requires_grad=False)
        return head
    return made


HEADS = {"subclass": lambda head: Doubled(1024, 8192, bias=False).cuda().half(), "hook": hooked, "bias": with_bias,
         "weight of a subclass": with_weight(lambda w: w.as_subclass(Marked)), "strided": with_weight(lambda w: w.t().contiguous().t()), "off the grid": with_weight(lambda w: off_by_one(w)),
         "row length": with_weight(lambda w: torch.cat([w, w[:, :128]], 1).contiguous()),
         "fewer rows than pay": with_weight(lambda w: w[:8191].contiguous()), "shorter rows than pay": with_weight(lambda w: w[:, :768].contiguous())}


@pytest.mark.parametrize("rows", [1, 2, 7, 16, 17])
@pytest.mark.parametrize("kind", [None, *HEADS])
def test_which_lm_heads_the_kernel_computes(monkeypatch, kind, rows):
    """Up to 16 rows of torch's own linear layer with nothing hung on it and enough of a weight: the kernel, once.  Everything else:
    the module, whose result comes back as it is."""
    from gptq_triton_amd import llama
    calls = []
    real = llama.lm_head_logits
    monkeypatch.setattr(llama, "lm_head_logits", lambda x, w: calls.append(1) or real(x, w))
    model = llama.LlamaForCausalLM.__new__(llama.LlamaForCausalLM)
    torch.nn.Module.__init__(model)
    head = torch.nn.Linear(1024, 8192, bias=False).cuda().half()
    model.lm_head = head if kind is None else HEADS[kind](head)
    h = torch.randn((rows, 1, model.lm_head.weight.shape[1]), device="cuda").half()
    with torch.no_grad():
        got, want = model._logits(h), model.lm_head(h)
    assert len(calls) == (kind is None and rows <= 16)
    if calls:   # (either rounds its fp32 sums to fp16 once)
        assert float((got.float() - want.float()).abs().max()) <= 2.0 ** -10 * float(want.abs().max())
    else:
        assert torch.equal(got, want)
