"""The two non-matmul operators of a decode step, as HIP kernels behind the C ABI: RMSNorm
and single-query attention over a preallocated KV cache.  The reference runs both as torch
ops of the HF model it patches (LlamaRMSNorm; fused_attention.py:118-148); here they exist
so that a whole decode step is a short chain of HIP launches that a graph can replay."""
from __future__ import annotations

import os

import torch

from . import _lib


# limits of the matmul kernels that normalise their own input (gptq4_norm_qkv_rotary, gptq4_norm_mlp_gateup)
NORM_MAX_ROWS, NORM_MAX_HIDDEN = 4, 8192
# up to how many rows the decoder uses them on weights in checkpoint order: one row costs 1.3-1.4 us on top of the plain
# projection against a 2.8 us norm launch; two rows about as much as the launch, three and four more (every workgroup
# normalises every row, one after the other).  In streaming order (norm_fusion_pays: streamed) the rows are normalised side
# by side.  QKV and gate/up behind a norm launch / with the norm inside, weights from HBM, us:
#   hidden          1024                 4096                   5120                   6656                   8192
#   2 rows   7.5/6.3   6.9/5.7   10.9/9.0   14.5/12.2   14.7/12.6  19.5/16.9   20.3/17.7  27.8/24.8   25.5/22.9  37.8/34.8
#   3 rows   7.6/6.7   7.2/6.1   11.7/9.9   14.9/13.0   13.7/12.6  19.2/18.0   19.6/18.0  27.9/26.4   24.5/23.0  38.2/36.5
#   4 rows   7.8/7.2   7.3/6.6   11.8/10.5  14.9/13.6   14.0/13.4  19.6/18.6   19.9/19.0  28.1/27.2   25.5/23.5  38.7/36.6
# With act-order every workgroup also gathers the normalised rows, where the norm launch stores them in the order that is read:
#   3 rows   7.9/7.2   7.5/6.6   12.1/10.8  15.4/14.0   14.1/13.7  19.8/19.1   20.1/19.4  28.4/27.6   24.8/24.7  38.6/37.9
#   4 rows   8.1/7.8   7.5/7.2   12.2/11.6  15.4/14.8   14.4/14.7  20.1/20.1   20.4/20.7  28.7/29.0   25.9/25.7  39.0/38.9
NORM_PAYS_ROWS = 1
# so four act-order rows take the norm along up to this hidden size (4352: 13.1/13.3  16.9/16.8, 7168: 21.7/22.3  31.6/31.1)
NORM_PAYS_GATHERED = 4096
# GPTQ4_NORM_FUSION=0 in the environment keeps the norms as launches of their own (for A/B timing)
NORM_FUSION = os.environ.get("GPTQ4_NORM_FUSION", "1") != "0"


def norm_fusable(rows: int, hidden: int) -> bool:
    """Whether a projection of `rows` rows CAN take the residual add + RMSNorm of its input along."""
    return 0 < rows <= NORM_MAX_ROWS and hidden <= NORM_MAX_HIDDEN and hidden % 8 == 0


def norm_fusion_pays(rows: int, hidden: int, streamed=None) -> bool:
    """Whether it is also the faster way (what the decoder asks).  streamed(): the rows that the launch on streaming-order
    weights normalises, 0 in checkpoint order, and whether it gathers them afterwards (act-order)."""
    if not (NORM_FUSION and norm_fusable(rows, hidden)):
        return False
    if rows <= NORM_PAYS_ROWS or NORM_PAYS_ROWS == 0 or streamed is None:
        return rows <= NORM_PAYS_ROWS
    most, gathers = streamed()
    return rows <= most and not (gathers and rows == NORM_MAX_ROWS and hidden > NORM_PAYS_GATHERED)


def check_norm_args(h: torch.Tensor, delta, weight: torch.Tensor):
    """Say what is wrong with (h, delta, norm weight) of a fused call."""
    for t, name in ((h, "h"), (delta, "delta"), (weight, "norm weight")):
        if t is None:
            continue
        _lib.require_cuda(t, name)
        if t.dtype != torch.float16:
            raise TypeError("the fused residual add + RMSNorm takes fp16 tensors")
    hidden = h.shape[-1]
    if weight.shape != (hidden,) or (delta is not None and delta.shape != h.shape):
        raise ValueError("h and delta must have one shape [..., H] and the norm weight [H]")


def contiguous_delta(delta):
    """The residual of a fused call as the kernels read it (a strided one is copied; None stays None)."""
    return delta if delta is None or delta.is_contiguous() else delta.contiguous()


def _check_out_index(out_index, h: int) -> None:
    if out_index is not None:
        _lib.require_cuda(out_index, "out_index")
        if out_index.dtype != torch.int32 or out_index.shape != (h,) or not out_index.is_contiguous():
            raise ValueError(f"out_index must be a contiguous int32 tensor of {h} positions")


def rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float, out_index: torch.Tensor = None) -> torch.Tensor:
    """y = weight * fp16(x * rsqrt(mean(x^2, -1) + eps)) for fp16 x [..., H] on the GPU.  With out_index (int32
    [H], a permutation) value f of a row is stored at position out_index[f]."""
    y = _lib.host().rms_norm(x, weight, eps, out_index)
    if y is not None:
        return y
    _lib.require_cuda(x, "x")
    _lib.require_cuda(weight, "weight")
    if x.dtype != torch.float16 or weight.dtype != torch.float16:
        raise TypeError("rms_norm takes fp16 tensors")
    h = x.shape[-1]
    if weight.shape != (h,) or h % 8 != 0:
        raise ValueError(f"weight must be [{h}] and the hidden size a multiple of 8")
    _check_out_index(out_index, h)
    if x.is_contiguous() and weight.is_contiguous():
        raise _lib.refused("rms_norm")
    return rms_norm(x.contiguous(), weight.contiguous(), eps, out_index)


def add_rms_norm(x: torch.Tensor, delta: torch.Tensor, weight: torch.Tensor, eps: float, out_index: torch.Tensor = None):
    """(x + delta, RMSNorm(x + delta)) in one launch; fp16 GPU tensors of equal shape [..., H].  out_index as in
    rms_norm (the sum keeps its order)."""
    both = _lib.host().add_rms_norm(x, delta, weight, eps, out_index)
    if both is not None:
        return both
    for t, name in ((x, "x"), (delta, "delta"), (weight, "weight")):
        _lib.require_cuda(t, name)
        if t.dtype != torch.float16:
            raise TypeError("add_rms_norm takes fp16 tensors")
    h = x.shape[-1]
    if delta.shape != x.shape or weight.shape != (h,) or h % 8 != 0:
        raise ValueError("x and delta must have one shape [..., H], weight [H], H a multiple of 8")
    _check_out_index(out_index, h)
    if x.is_contiguous() and delta.is_contiguous() and weight.is_contiguous():
        raise _lib.refused("add_rms_norm")
    return add_rms_norm(x.contiguous(), delta.contiguous(), weight.contiguous(), eps, out_index)


HEAD_MAX_ROWS = 16


def head_argmax_takes(rows: int, weight: torch.Tensor) -> bool:
    """Whether the lm_head kernels take this many rows for an fp16 weight [V, K] (which they read 16 bytes at a time; x lies in LDS)."""
    k = weight.shape[1]
    return weight.is_cuda and weight.dtype == torch.float16 and weight.is_contiguous() and weight.data_ptr() % 16 == 0 \
        and k % 256 == 0 and 0 < rows <= HEAD_MAX_ROWS \
        and rows * (k + 8) * 2 <= 160 * 1024 - 2048 and weight.numel() * 2 < 0x7FFFFFF0


def head_logits_pays(rows: int, weight: torch.Tensor) -> bool:
    """Whether lm_head_logits is the faster way to rows of logits.  Against torch's product, us, from HBM, at 1 / 8 / the most rows:
    32000 x 1024 13.3 / 14.3 / 16.0 to 17.3 / 17.5 / 17.9, x 4096 46.1 / 45.9 / 47.6 to 62.6 / 61.4 / 61.3,
    x 5120 54.9 / 54.3 / 56.9 to 66.2 / 63.7 / 64.2, x 6656 69.7 / 68.6 / 69.9 to 83.7 / 80.6 / 80.9, x 8192 84.5 / 84.8 / 85.4 to 99.1 / 97.4 / 97.3;
    8192 x 2048 8.5 / 9.6 / 10.3 to 13.1 / 13.3 / 13.5, x 8192 25.3 / 26.8 / 27.1 to 31.4 / 30.5 / 30.3; 50304 x 1024 20.8 / 21.1 / 23.3 to 23.3 / 22.8 / 23.6.
    Not with few of either: 4096 x 8192 16.2 / 17.7 / 18.0 to 16.1 / 16.3 / 16.3, 320 x 6656 10.0 / 11.5 / 12.3 to 8.1 / 8.2 / 8.2 (every
    workgroup brings all of x into its LDS), 50304 x 768 18.5 / 18.8 / 20.8 to 19.4 / 19.1 / 19.7."""
    return weight.shape[0] >= 8192 and weight.shape[1] >= 1024 and head_argmax_takes(rows, weight)


def lm_head_argmax(x: torch.Tensor, weight: torch.Tensor, max_rows: int = HEAD_MAX_ROWS) -> torch.Tensor:
    """Greedy next tokens: argmax(x @ weight.T, -1) in one launch, for x fp16 [..., K] and an fp16 lm_head weight [V, K].
    Returns int64 of x's shape without the last dimension.  More than `max_rows` rows, and shapes the kernel does not take
    (head_argmax_takes), go through torch."""
    k = x.shape[-1]
    rows = x.numel() // max(k, 1)
    if rows > max_rows or weight.dim() != 2 or weight.shape[1] != k or not x.is_cuda or x.dtype != torch.float16 or not head_argmax_takes(rows, weight):
        return torch.nn.functional.linear(x, weight).argmax(-1)
    x = x.contiguous()
    out = _lib.host().lm_head_argmax(x if x.data_ptr() % 16 == 0 else x.clone(), weight)
    if out is None:
        raise _lib.refused("lm_head_argmax")
    return out


def lm_head_logits(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """x @ weight.T for the rows of x fp16 [..., K] and the fp16 lm_head weights [V, K] that head_argmax_takes: up to HEAD_MAX_ROWS, and
    no more than fit the LDS (15 of 5120 values, 12 of 6656, 9 of 8192)."""
    x = x.contiguous()
    out = _lib.host().lm_head_logits(x if x.data_ptr() % 16 == 0 else x.clone(), weight)
    if out is None:
        raise _lib.refused("lm_head_logits")
    return out


def greedy_step_end(x, delta, norm_weight, eps, weight, tokens, positions, history, embed=None, next_hidden=None) -> None:
    """The end of a greedy decode step in one launch: tokens (int64) become the argmax of the logits, positions (int32) go up by
    one, the tokens are stored at those places of history (int64 [B, capacity]) and, if given, their rows of the embedding in
    next_hidden.
    norm_weight None: x is what the lm_head reads; else (one row) x is the residual stream and the logits are those of
    RMSNorm(x + delta) * norm_weight, as add_rms_norm gives it."""
    if _lib.host().greedy_step_end(x, delta, norm_weight, eps, weight, tokens, positions, history, embed, next_hidden) is None:
        raise _lib.refused("greedy_step_end")


def prefill_attention(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, past: int = 0) -> torch.Tensor:
    """Causal attention of a prompt (or of a chunk behind `past` cached tokens): q fp16 [B, H, S, 128]; caches fp16
    [B, H, capacity, 128] holding the S new tokens in rows past .. past + S - 1 (for a plain prompt: the k and v the QKV
    projection returned); query i attends to rows 0 .. past + i.  Returns fp16 [B, S, H*128], what o_proj consumes."""
    out = _lib.host().prefill_attention(q, k_cache, v_cache, past)
    if out is not None:
        return out
    for t, name in ((q, "q"), (k_cache, "k_cache"), (v_cache, "v_cache")):
        _lib.require_cuda(t, name)
        if t.dtype != torch.float16:
            raise TypeError("prefill_attention takes fp16 tensors")
    bsz, heads, q_len, hd = q.shape
    if hd != 128:
        raise ValueError("prefill_attention needs head_dim 128")
    if k_cache.shape != v_cache.shape or k_cache.shape[:2] != (bsz, heads) or k_cache.shape[3] != hd \
            or not (q.is_contiguous() and k_cache.is_contiguous() and v_cache.is_contiguous()):
        raise ValueError("caches must be contiguous [B, H, capacity, 128] tensors matching q")
    cap = k_cache.shape[2]
    if past < 0 or past + q_len > cap:
        raise ValueError("the cache has no room for past + S rows")
    raise _lib.refused("prefill_attention")


def decode_attention(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, positions: torch.Tensor,
                     out_index: torch.Tensor = None) -> torch.Tensor:
    """q fp16 [B, H, 1, 128]; caches fp16 [B, H, capacity, 128]; positions int32 [B] or [B, 1]:
    sequence b attends to cache rows 0..positions[b].  Returns fp16 [B, 1, H*128]; with out_index
    (int32 [H*128], a permutation) feature f of a row is stored at position out_index[f]."""
    out = _lib.host().decode_attention(q, k_cache, v_cache, positions, out_index)
    if out is not None:
        return out
    for t, name in ((q, "q"), (k_cache, "k_cache"), (v_cache, "v_cache"), (positions, "positions")):
        _lib.require_cuda(t, name)
    bsz, heads, q_len, hd = q.shape
    if q_len != 1 or hd != 128:
        raise ValueError("decode_attention takes one query token per sequence and head_dim 128")
    if k_cache.shape != v_cache.shape or k_cache.shape[:2] != (bsz, heads) or k_cache.shape[3] != hd \
            or not (q.is_contiguous() and k_cache.is_contiguous() and v_cache.is_contiguous()):
        raise ValueError("caches must be contiguous [B, H, capacity, 128] tensors matching q")
    if q.dtype != torch.float16 or k_cache.dtype != torch.float16 or v_cache.dtype != torch.float16:
        raise TypeError("decode_attention takes fp16 tensors")
    if positions.numel() != bsz:
        raise ValueError("one position per sequence")
    _check_out_index(out_index, heads * hd)
    if positions.dtype == torch.int32 and positions.is_contiguous():
        raise _lib.refused("decode_attention")
    return decode_attention(q, k_cache, v_cache, positions.to(torch.int32).contiguous(), out_index)


ATTENTION_MAX_HEADS = 4096  # sequences x heads of one decode_attention / extend_attention call


def extend_attention(q: torch.Tensor, past_k, past_v, k: torch.Tensor, v: torch.Tensor, out_index: torch.Tensor = None) -> torch.Tensor:
    """One query token per sequence over a (key, value) pair that grows by a row: q fp16 [B, H, 1, 128]; past_k, past_v fp16
    [B, H, past, 128] (None: no past); k, v [B, H, past + 1, 128], whose last row is in place already - the other rows are
    copied from the past on the way.  Attends to all past + 1 rows; result and out_index as in decode_attention."""
    out = _lib.host().extend_attention(q, past_k, past_v, k, v, out_index)
    if out is not None:
        return out
    for t, name in ((q, "q"), (past_k, "past_k"), (past_v, "past_v"), (k, "k"), (v, "v")):
        if t is not None:
            _lib.require_cuda(t, name)
    _check_out_index(out_index, q.shape[1] * q.shape[3])
    raise ValueError("extend_attention takes contiguous fp16 tensors: q [B, H, 1, 128], past [B, H, P, 128], k and v [B, H, P + 1, 128]")
