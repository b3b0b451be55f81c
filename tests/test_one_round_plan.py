"""Calls of more than 16 rows that the planner sends to the mid-M kernel in one round of workgroups by its estimated time: the range
of that rule (host arithmetic), and parity at automatic plans, narrow widths and more than 768 rows among them."""
import numpy as np
import pytest
import torch

from gptq_triton_amd import _lib

MATMUL, GATEUP, QKV = 0, 1, 2


def planned(op, m, k, n):
    return _lib.load().gptq4_planned_kernel(op, m, k, n)


def test_calls_that_were_timed_slower_are_not_planned_by_the_estimate():
    for op, m, k, n in [(0, 512, 512, 6144), (0, 1024, 512, 4096), (0, 512, 768, 6144), (1, 1280, 512, 1536), (1, 192, 512, 3072),  # short rows
                        (0, 4096, 5120, 512), (0, 8192, 5120, 256), (0, 8192, 512, 512), (1, 4096, 2048, 512),                     # many rows
                        (1, 2048, 11008, 1024), (1, 2048, 16384, 1024), (1, 1024, 16384, 1536), (0, 1024, 2048, 4096)]:            # 5 % ahead only
        assert planned(op, m, k, n) != 2, (op, m, k, n)


def test_calls_that_were_timed_faster_still_are():
    for op, m, k, n in [(0, 96, 4096, 4096), (1, 96, 4096, 11008), (0, 192, 4096, 12288), (0, 640, 4096, 4096),
                        (0, 64, 512, 4096), (2, 512, 512, 1536), (0, 800, 4096, 1024), (0, 2048, 4096, 512), (2, 1536, 1024, 768),
                        (1, 800, 4096, 1024)]:
        assert planned(op, m, k, n) == 2, (op, m, k, n)


def test_the_rule_ends_at_8192_rows_and_other_calls_have_no_answer():
    assert all(planned(op, m, k, n) != 2 for op in (0, 1, 2) for m in (8193, 16384) for k in (1024, 4096) for n in (256 if op < 2 else 768,))
    assert planned(0, 16, 4096, 4096) < 0 and planned(0, 64, 4096, 4000) < 0 and planned(3, 64, 4096, 4096) < 0


SHAPES = [(MATMUL, 17, 4096, 1024), (MATMUL, 64, 512, 4096), (MATMUL, 65, 1024, 1024), (MATMUL, 768, 1024, 1024), (MATMUL, 769, 1024, 1024),
          (MATMUL, 1100, 2048, 768), (MATMUL, 2048, 4096, 512), (MATMUL, 2049, 4096, 256), (MATMUL, 97, 4096, 1280),
          (GATEUP, 17, 4096, 1024), (GATEUP, 65, 2048, 768), (GATEUP, 769, 4096, 1024), (GATEUP, 1501, 4096, 256), (GATEUP, 320, 1024, 768),
          (QKV, 33, 1024, 1536), (QKV, 65, 1024, 1536), (QKV, 513, 512, 1536), (QKV, 801, 1024, 768), (QKV, 1537, 1024, 768)]


@pytest.mark.gpu
@pytest.mark.parametrize("stream", [False, True])
@pytest.mark.parametrize("op,m,k,n", SHAPES)
def test_automatic_plans_agree_with_the_decode_kernels(op, m, k, n, stream):
    """Every row as the kernels for up to 16 rows compute it, up to the rounding to fp16 and the order of the fp32 sums: with S the
    sum of |x w| behind a value, each side's sum is within K 2^-24 S of the exact one."""
    import gptq_triton_amd as G
    from gptq_triton_amd import fused_attention as A, fused_mlp as F, quant_linear as Q
    if stream and Q.stream_rows(op, k, n, 128) < 16:
        pytest.skip("no streaming order for this shape")
    assert planned(op, m, k, n) == 2
    gen = torch.Generator(device="cuda").manual_seed(m + k + n + op)
    words = lambda *s: torch.randint(-2 ** 31, 2 ** 31 - 1, s, dtype=torch.int32, device="cuda", generator=gen)
    g = 128

    def matrix():
        w, z = words(k // 8, n), words(k // g, n // 8)
        s = ((0.2 + 0.3 * torch.rand((k // g, n), device="cuda", generator=gen)) / (4.6 * k ** 0.5)).half()
        return w, s, z

    mats = [matrix() for _ in range(2 if op == GATEUP else 1)]
    x = torch.randn((m, k), device="cuda", generator=gen).half()
    packed = [Q.stream_pack(w, z, s, g) for w, s, z in mats] if stream else None
    cos, sin = G.RotaryTable(128, 4096).get(x.device, 4096)
    pos = torch.arange(m, dtype=torch.int32, device="cuda")

    def run(rows):
        a = x[rows]
        if op == MATMUL:
            return Q.matmul4_stream(g, a, *packed[0]) if stream else Q.matmul4(g, a, *mats[0])
        if op == GATEUP:
            return F.llama_mlp_4_stream(g, a, *packed[0], *packed[1]) if stream else F.llama_mlp_4(g, a, *mats[0], *mats[1])
        p, heads = pos[rows][None], n // 384
        out = A.qkv_rotary_stream(g, a[None], *packed[0], p, cos, sin, heads, 128) if stream \
            else A.qkv_rotary(g, a[None], *mats[0], p, cos, sin, heads, 128)
        return torch.cat([t[0].transpose(0, 1).reshape(a.shape[0], -1) for t in out], dim=1)

    got = run(slice(0, m))
    assert torch.equal(got, run(slice(0, m))), "the reduction order is fixed"
    want = torch.cat([run(slice(i, min(i + 16, m))) for i in range(0, m, 16)])
    dense = [Q.dequantize(w, z, s, g).float() for w, s, z in mats]
    sums = [x.abs().float() @ d.abs() for d in dense]
    order = 2 * k * 2.0 ** -24
    if op == MATMUL:
        slack = order * sums[0]
    elif op == GATEUP:      # |silu'| <= 1.1
        up, gate = x.float() @ dense[1], x.float() @ dense[0]
        slack = order * (1.1 * sums[0] * (up.abs() + 1) + sums[1] * gate.abs())
    else:                   # a rotated value is a sum of two products with |cos|, |sin| <= 1
        slack = order * 2 * sums[0].amax(1, keepdim=True)
    big = torch.maximum(got.abs(), want.abs()).cpu().numpy()
    ulp = torch.from_numpy(np.spacing(big).astype(np.float32)).cuda()
    worst = ((got.float() - want.float()).abs() - ulp - slack).max().item()
    assert worst <= 0.0, worst


# (rows, inputs, outputs, act-order, bytes of workspace behind its head): the plan by scores fits, the one by estimated time does not
TIGHT = [(70, 12672, 6400, False, 0), (84, 13696, 12800, False, 8 << 20), (76, 19456, 10240, False, 4 << 20), (191, 6912, 5632, True, 4 << 20)]


def matmul_in(workspace, tensors, m, k, n):
    """The library's return code of a call with that (address, bytes) of workspace."""
    x, w, z, s, perm, y = tensors
    stream = 0 if not torch.cuda.is_available() else torch.cuda.current_stream().cuda_stream
    return _lib.load().gptq4_matmul(x, w, z, s, perm, None, y, m, k, n, 128, *workspace, stream)


@pytest.mark.skipif(torch.cuda.is_available(), reason="the addresses are not memory: without a GPU nothing is launched")
def test_a_workspace_that_the_plan_by_scores_fits_is_enough():
    fake = 4096
    for m, k, n, act_order, extra in TIGHT:
        rc = matmul_in((fake, _lib.WS_HEAD_BYTES + extra), (fake, fake, fake, fake, fake if act_order else None, fake), m, k, n)
        assert rc > 0, (rc, m, k, n)                    # (HIP's: there is no device)
    for m, k, n in [(646, 14720, 22784), (677, 17152, 22784), (711, 13184, 22784)]:
        rc = _lib.load().gptq4_matmul_static(fake, fake, fake, fake, None, fake, m, k, n, 128, None)
        assert rc > 0, (rc, m, k, n)


@pytest.mark.gpu
@pytest.mark.parametrize("m,k,n,act_order,extra", TIGHT)
def test_calls_with_a_tight_workspace(m, k, n, act_order, extra):
    """As with all the workspace the library asks for, up to the order of the fp32 sums (see above)."""
    from gptq_triton_amd import quant_linear as Q
    gen = torch.Generator(device="cuda").manual_seed(m)
    words = lambda *s: torch.randint(-2 ** 31, 2 ** 31 - 1, s, dtype=torch.int32, device="cuda", generator=gen)
    w, z = words(k // 8, n), words(k // 128, n // 8)
    s = ((0.2 + 0.3 * torch.rand((k // 128, n), device="cuda", generator=gen)) / (4.6 * k ** 0.5)).half()
    x = torch.randn((m, k), device="cuda", generator=gen).half()
    perm = torch.randperm(k, device="cuda", generator=gen).int() if act_order else None
    ws = torch.zeros(_lib.WS_HEAD_BYTES + extra, dtype=torch.uint8, device="cuda")
    got = torch.empty((m, n), dtype=torch.float16, device="cuda")
    rc = matmul_in((ws.data_ptr(), ws.numel()), (x.data_ptr(), w.data_ptr(), z.data_ptr(), s.data_ptr(), _lib.ptr(perm), got.data_ptr()), m, k, n)
    assert rc == 0
    want = Q.matmul4(128, x, w, s, z, perm=perm)
    ordered = x if perm is None else x[:, perm.long()]
    slack = 2 * k * 2.0 ** -24 * (ordered.abs().float() @ Q.dequantize(w, z, s, 128).abs().float())
    ulp = torch.from_numpy(np.spacing(torch.maximum(got.abs(), want.abs()).cpu().numpy()).astype(np.float32)).cuda()
    assert ((got.float() - want.float()).abs() - ulp - slack).max().item() <= 0.0
    assert int(ws[:_lib.WS_HEAD_BYTES].view(torch.int32).abs().sum()) == 0
