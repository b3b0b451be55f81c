"""A minimal LLaMA decoder around the quantised hot path.

The reference builds an un-initialised HF `LlamaForCausalLM` and swaps modules in it
(src/gptq_triton/__init__.py:32-77); generation is then HF's (generate.py:41-50).  Here the
model skeleton is a few lines of plain torch with the same module tree and therefore the
same state_dict keys (`model.layers.{i}.self_attn.q_proj.qweight`, ...), so reference
checkpoints load unchanged and nothing depends on transformers at run time.  RMSNorm,
residuals, the attention core and the fp16 lm_head are torch ops; every linear inside the
layers is the HIP path.
"""
from __future__ import annotations

import json
from pathlib import Path
from typing import List, Optional, Tuple

import torch
import torch.nn as nn

from . import _lib
from .decoder_ops import (NORM_MAX_HIDDEN, add_rms_norm, decode_attention, greedy_step_end, head_argmax_takes, head_logits_pays, lm_head_argmax,
                          lm_head_logits, norm_fusion_pays, prefill_attention, rms_norm)
from .fused_attention import KV_AT_POSITION, LlamaConfigLite, QuantLlamaAttention
from .fused_mlp import QuantLlamaMLP, llama_mlp_4_stream
from .quant_linear import InverseOrder, QuantLinear, child, only_itself, plain_module, stream_norm_rows, stream_rows

# the rows the decode kernels built on the streaming-order weight layout take (more rows: the mid-M and tiled kernels)
STREAM_BATCH = 16
LINEAR_FORWARD = nn.Linear.forward  # torch's own


def config_from_json(path) -> LlamaConfigLite:
    """Read the fields this path needs from an HF-style config.json."""
    raw = json.load(open(path))
    cfg = LlamaConfigLite()
    for field in ("hidden_size", "num_attention_heads", "max_position_embeddings", "rope_theta", "intermediate_size",
                  "num_hidden_layers", "vocab_size", "rms_norm_eps"):
        if field in raw:
            setattr(cfg, field, raw[field])
    kv = raw.get("num_key_value_heads", cfg.num_attention_heads)
    if kv != cfg.num_attention_heads:
        raise NotImplementedError("grouped-query attention is outside the LLaMA-1 family this path covers")
    return cfg


class LlamaRMSNorm(nn.Module):
    def __init__(self, hidden_size: int, eps: float = 1e-6):
        super().__init__()
        self.weight = nn.Parameter(torch.ones(hidden_size, dtype=torch.float16), requires_grad=False)
        self.variance_epsilon = eps

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        if x.is_cuda and x.dtype == torch.float16:
            return rms_norm(x, self.weight, self.variance_epsilon)  # one HIP launch
        xf = x.float()
        xf = xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + self.variance_epsilon)
        return self.weight * xf.to(x.dtype)

    own_forward = forward


class LlamaAttention(nn.Module):
    """Skeleton attention block: four linears to be replaced by make_quant / make_quant_attn."""

    def __init__(self, config):
        super().__init__()
        self.config = config
        h = config.hidden_size
        self.q_proj = nn.Linear(h, h, bias=False)
        self.k_proj = nn.Linear(h, h, bias=False)
        self.v_proj = nn.Linear(h, h, bias=False)
        self.o_proj = nn.Linear(h, h, bias=False)


class LlamaMLP(nn.Module):
    """Skeleton MLP block: three linears to be replaced by make_quant / make_fused_mlp."""

    def __init__(self, config):
        super().__init__()
        h, i = config.hidden_size, config.intermediate_size
        self.gate_proj = nn.Linear(h, i, bias=False)
        self.down_proj = nn.Linear(i, h, bias=False)
        self.up_proj = nn.Linear(h, i, bias=False)
        self._same_rows = InverseOrder()  # of gate's and up's permutation, where it is one
        self._most_rows = (None, 0)  # (sizes, rows): see _pair_rows

    def _pair(self, rows: int):
        """(groupsize, gate words and {scale, zero} words, up's, row permutation) where one launch can compute
        silu(gate) * up from the two modules' own tensors in streaming order, else None."""
        gate, up = child(self, 'gate_proj'), child(self, 'up_proj')
        if not (only_itself(gate, QuantLinear) and only_itself(up, QuantLinear)):
            return None
        g, u = gate.stream_weights(rows), up.stream_weights(rows)
        if g is None or u is None or gate.groupsize != up.groupsize or g[0].shape != u[0].shape \
                or gate.bias_tensor() is not None or up.bias_tensor() is not None or rows <= 16 and self._pair_rows(gate) < rows:
            return None
        if (g[2] is None) != (u[2] is None) or g[2] is not None and self._same_rows.of(g[2], u[2]) is None:
            return None
        return gate.groupsize, g[0], g[1], u[0], u[1], g[2]

    def input_order(self):
        """As QuantLlamaMLP.input_order: None without act-order, where gate and up each have an order of their own, and where
        this block, gate or up is to be called as a module (only_itself)."""
        gate, up = child(self, 'gate_proj'), child(self, 'up_proj')
        if not (only_itself(self, LlamaMLP) and only_itself(gate, QuantLinear) and only_itself(up, QuantLinear)) \
                or gate.g_idx is None or up.g_idx is None:
            return None
        return self._same_rows.of(gate.row_permutation(), up.row_permutation())

    def _pair_rows(self, gate) -> int:
        sizes = gate.infeatures, gate.outfeatures, gate.groupsize
        if self._most_rows[0] != sizes:
            self._most_rows = sizes, stream_rows(_lib.OP_MLP_GATEUP, *sizes)
        return self._most_rows[1]

    def forward(self, x, ordered: bool = False):
        # without make_fused_mlp the three projections stay modules of their own; on the GPU gate and up still are one
        # launch, with SiLU and the product on the fp32 sums (two launches and two elementwise ones otherwise)
        pair = self._pair(x.numel() // max(x.shape[-1], 1)) if x.is_cuda else None
        if pair is not None:
            groupsize, gw, gm, uw, um, perm = pair
            return child(self, 'down_proj')(llama_mlp_4_stream(groupsize, x, gw, gm, uw, um, None if ordered else perm))
        if ordered:
            return self.down_proj(torch.nn.functional.silu(self.gate_proj.multiply(x, ordered=True)) * self.up_proj.multiply(x, ordered=True))
        return self.down_proj(torch.nn.functional.silu(self.gate_proj(x)) * self.up_proj(x))

    own_forward = forward

    def norm_fusable(self, rows: int) -> bool:
        """Whether forward_normed is the faster way for this many rows."""
        gate = child(self, 'gate_proj')
        pair = self._pair(rows) if only_itself(self, LlamaMLP) else None
        return pair is not None and norm_fusion_pays(rows, gate.infeatures, lambda: (
            stream_norm_rows(_lib.OP_MLP_GATEUP, gate.infeatures, gate.outfeatures, gate.groupsize), pair[5] is not None))

    def forward_normed(self, h, delta, norm_weight, eps):
        """(h + delta, forward(RMSNorm(h + delta))) with the residual add and the norm inside the gate/up launch."""
        groupsize, gw, gm, uw, um, perm = self._pair(h.numel() // h.shape[-1])
        s, mid = llama_mlp_4_stream(groupsize, h, gw, gm, uw, um, perm, norm=(delta, norm_weight, eps))
        return s, child(self, 'down_proj')(mid)


class LlamaDecoderLayer(nn.Module):
    def __init__(self, config):
        super().__init__()
        self.self_attn = LlamaAttention(config)
        self.mlp = LlamaMLP(config)
        self.input_layernorm = LlamaRMSNorm(config.hidden_size, config.rms_norm_eps)
        self.post_attention_layernorm = LlamaRMSNorm(config.hidden_size, config.rms_norm_eps)

    def forward(self, hidden_states, attention_mask=None, position_ids=None, past_key_value=None, use_cache=False, causal=False):
        attn_out, _, present = self.self_attn(hidden_states=self.input_layernorm(hidden_states),
                                              attention_mask=attention_mask, position_ids=position_ids,
                                              past_key_value=past_key_value, use_cache=use_cache, causal=causal)
        hidden_states = hidden_states + attn_out
        hidden_states = hidden_states + self.mlp(self.post_attention_layernorm(hidden_states))
        return hidden_states, present

    own_forward = forward

    def only_themselves(self) -> bool:
        """Whether the layer and the blocks it calls are this package's own and nothing else would run with them."""
        attn, mlp = child(self, 'self_attn'), child(self, 'mlp')
        return only_itself(self, LlamaDecoderLayer) and only_itself(attn, QuantLlamaAttention) \
            and only_itself(mlp, QuantLlamaMLP if type(mlp) is QuantLlamaMLP else LlamaMLP) \
            and only_itself(child(self, 'input_layernorm'), LlamaRMSNorm) \
            and only_itself(child(self, 'post_attention_layernorm'), LlamaRMSNorm)


class LlamaModel(nn.Module):
    def __init__(self, config):
        super().__init__()
        self.embed_tokens = nn.Embedding(config.vocab_size, config.hidden_size)
        self.layers = nn.ModuleList([LlamaDecoderLayer(config) for _ in range(config.num_hidden_layers)])
        self.norm = LlamaRMSNorm(config.hidden_size, config.rms_norm_eps)


def causal_mask(q_len: int, kv_len: int, device, dtype=torch.float16) -> Optional[torch.Tensor]:
    """Additive [1, 1, q_len, kv_len] mask; None when a single query row sees everything."""
    if q_len == 1:
        return None
    past = kv_len - q_len
    i = torch.arange(q_len, device=device)[:, None]
    j = torch.arange(kv_len, device=device)[None, :]
    m = torch.zeros((q_len, kv_len), dtype=dtype, device=device)
    m.masked_fill_(j > i + past, torch.finfo(dtype).min)
    return m[None, None]


class LlamaForCausalLM(nn.Module):
    def __init__(self, config):
        super().__init__()
        self.config = config
        self.model = LlamaModel(config)
        self.lm_head = nn.Linear(config.hidden_size, config.vocab_size, bias=False)
        self.seqlen = config.max_position_embeddings

    @torch.no_grad()
    def forward(self, input_ids: torch.Tensor, past_key_values: Optional[List[Tuple[torch.Tensor, torch.Tensor]]] = None,
                use_cache: bool = False, last_token_only: bool = False):
        """input_ids [B, S] -> (logits [B, S or 1, vocab], past_key_values or None)."""
        bsz, q_len = input_ids.shape
        past_len = 0 if past_key_values is None else past_key_values[0][0].shape[2]
        h = self.model.embed_tokens(input_ids)
        layers = self.model.layers
        if h.is_cuda and h.dtype == torch.float16 and len(layers) and only_itself(self.model.norm, LlamaRMSNorm) \
                and all(type(l) is LlamaDecoderLayer and l.only_themselves() for l in layers):
            h, presents = self._layers_fused(h, past_len, past_key_values, use_cache)
            if last_token_only:
                h = h[:, -1:, :]
            return self._logits(h), (presents if use_cache else None)
        position_ids = torch.arange(past_len, past_len + q_len, device=input_ids.device).unsqueeze(0)
        presents = []
        for i, layer in enumerate(self.model.layers):
            # (causal: the attention block masks by position itself - on the GPU inside the attention kernel)
            h, present = layer(h, attention_mask=None, position_ids=position_ids,
                               past_key_value=None if past_key_values is None else past_key_values[i], use_cache=use_cache,
                               causal=True)
            presents.append(present)
        h = self.model.norm(h)
        if last_token_only:
            h = h[:, -1:, :]
        return self.lm_head(h), (presents if use_cache else None)

    def _logits(self, h):
        """lm_head(h); a few rows in a launch of this package's where that is faster (head_logits_pays), lm_head is torch's own linear
        layer and nothing else would run with it."""
        head = self.lm_head
        if type(head) is nn.Linear and plain_module(head) and nn.Linear.forward is LINEAR_FORWARD and head.bias is None:
            weight = head.weight
            # (a tensor subclass may stand for other values than those at its address)
            if type(weight) in (nn.Parameter, torch.Tensor) and weight.device == h.device and weight.dim() == 2 \
                    and weight.shape[1] == h.shape[-1] and head_logits_pays(h.numel() // h.shape[-1], weight) \
                    and not torch.is_autocast_enabled(h.device.type):
                return lm_head_logits(h, weight)
        return head(h)

    def _layers_fused(self, h, past_len, past_key_values, use_cache):
        """The stack and the final norm with every residual add in the launch of the norm behind it, and with a
        few tokens in all both of them in the projection's launch (norm_fusion_pays)."""
        layers = self.model.layers
        bsz, q_len, _ = h.shape
        position_ids = layers[0].self_attn.rope.positions(h.device, past_len, bsz, q_len)
        inside = q_len == 1 and all(l.self_attn.norm_fusable(bsz) and l.mlp.norm_fusable(bsz) for l in layers)
        h = h.contiguous()  # (the projections that normalise their own input take no strides)
        presents = []
        delta = None
        for i, layer in enumerate(layers):
            attn, mlp = child(layer, 'self_attn'), child(layer, 'mlp')
            n1, n2 = child(layer, 'input_layernorm'), child(layer, 'post_attention_layernorm')
            past = None if past_key_values is None else past_key_values[i]
            if inside:
                context, present, h = attn.attend_one(h, position_ids, past, norm=(delta, norm_weight(n1), n1.variance_epsilon))
                h, delta = mlp.forward_normed(h, attn.project_out(*context), norm_weight(n2), n2.variance_epsilon)
            else:
                order = order_of(attn)
                if delta is None:
                    x = rms_norm(h, n1.weight, n1.variance_epsilon, out_index=order)
                else:
                    h, x = add_rms_norm(h, delta, n1.weight, n1.variance_epsilon, out_index=order)
                out, _, present = attn(hidden_states=x, position_ids=position_ids, past_key_value=past, use_cache=use_cache, causal=True,
                                       ordered=order is not None)
                order = order_of(mlp)
                h, x = add_rms_norm(h, out, n2.weight, n2.variance_epsilon, out_index=order)
                delta = mlp(x, ordered=True) if order is not None else mlp(x)
            presents.append(present if use_cache else None)
            del present  # (without use_cache a layer's pair is given back before the next one's is made)
        norm = self.model.norm
        return add_rms_norm(h, delta, norm.weight, norm.variance_epsilon)[1], presents

    @torch.no_grad()
    def generate_greedy(self, input_ids: torch.Tensor, max_new_tokens: int, use_graph: bool = False) -> torch.Tensor:
        """Prefill + greedy decode with a preallocated KV cache: the fused QKV kernel writes
        rotated K and V straight into the cache (no cat, no copies).  use_graph replays one
        captured HIP graph per decode token instead of launching the step's kernels one by
        one."""
        bsz, prompt = input_ids.shape
        dec = GreedyDecoder(self, bsz, prompt + max_new_tokens)
        first = dec.prefill(input_ids)
        rest = dec.decode(max_new_tokens - 1, use_graph=use_graph) if max_new_tokens > 1 else first[:, :0]
        return torch.cat([input_ids, first, rest], dim=1)


def norm_weight(norm: nn.Module) -> torch.Tensor:
    """A norm's weight as the launches that normalise their own input read it (a strided one is copied, as rms_norm does)."""
    w = norm.weight
    return w if w.is_contiguous() else w.contiguous()


def order_of(block):
    """Where the norm in front of an act-order block should store each feature (None: no act-order, or gathered by the block)."""
    fn = getattr(block, "input_order", None)
    return fn() if fn is not None else None


class GreedyDecoder:
    """Greedy generation state for one batch: KV caches of fixed capacity plus the static
    token / position buffers a decode step reads and writes.  Nothing in a decode step
    depends on a host-side value that changes from token to token (the QKV kernel places
    K and V by position id, the attention kernel reads how far to attend from the position
    buffer), so the step can be captured once as a HIP graph and replayed."""

    def __init__(self, model: LlamaForCausalLM, bsz: int, capacity: int, layout: str = 'auto'):
        """layout: 'stream' / 'checkpoint' put the model's packed weights into that layout first (quant_linear.set_layout;
        one copy either way), 'keep' leaves them as they are, 'auto' = 'stream': every kernel reads that layout, and the
        decode kernels for up to STREAM_BATCH rows are built on it."""
        cfg = model.config
        self.model, self.bsz, self.capacity = model, bsz, capacity
        dev = model.lm_head.weight.device
        if layout == 'auto':
            layout = 'stream'
        if layout != 'keep' and dev.type == 'cuda':
            from .quant_linear import set_layout
            set_layout(model, layout)
        heads, hd = cfg.num_attention_heads, cfg.hidden_size // cfg.num_attention_heads
        self.caches = [(torch.zeros((bsz, heads, capacity, hd), dtype=torch.float16, device=dev),
                        torch.zeros((bsz, heads, capacity, hd), dtype=torch.float16, device=dev))
                       for _ in model.model.layers]
        self.tokens = torch.zeros((bsz, 1), dtype=torch.long, device=dev)
        self.position = torch.zeros((bsz, 1), dtype=torch.int32, device=dev)
        self.history = torch.zeros((bsz, capacity + 1), dtype=torch.long, device=dev)
        self.graph = None
        self._graph_keeps_history = False  # whether the captured step is one with one_launch_end

    @property
    def one_launch_end(self) -> bool:
        """Whether a decode step ends in one launch that picks the tokens, moves the positions on and keeps the tokens at their
        places in `history`.  Asked for every step: the caller may replace or convert the lm_head of a decoder that is kept.
        (The launch can fetch the embedding rows of the next step too, but a step starts from `tokens`, which the caller may
        write to between two steps or two replays of `graph`.)"""
        head = self.model.lm_head
        return head_argmax_takes(self.bsz, head.weight) and getattr(head, "bias", None) is None

    def _layers(self, h, position_ids, kv_offset, attend, end):
        """The decoder stack on hidden states h [B, S, hidden]; every residual add is fused with the RMSNorm that follows it.
        Returns end(residual stream, its last addend, norm, None), or end(None, None, norm, normed hidden states) where the
        final norm has run: the greedy next tokens, for a decode step in place."""
        layers = self.model.model.layers
        rows = h.shape[0] * h.shape[1]
        if all(getattr(l.self_attn, "norm_fusable", lambda r: False)(rows) and getattr(l.mlp, "norm_fusable", lambda r: False)(rows)
               for l in layers):
            return self._layers_norm_in_matmul(h, position_ids, kv_offset, attend, end)
        # act-order: every norm writes in the order its consumer's sorted rows read, so the consumer needs no gather launch
        n0 = layers[0].input_layernorm
        oq = order_of(layers[0].self_attn)
        x = rms_norm(h, n0.weight, n0.variance_epsilon, out_index=oq)
        for i, (layer, (kc, vc)) in enumerate(zip(layers, self.caches)):
            attn = layer.self_attn
            q, _, _ = attn.project_qkv(x, position_ids, kv_out=(kc, vc), kv_offset=kv_offset, ordered=oq is not None)
            norm = layer.post_attention_layernorm
            om = order_of(layer.mlp)
            # attend -> ([B, S, hidden], whether in attn.context_order())
            h, x = add_rms_norm(h, attn.project_out(*attend(q, kc, vc, attn)), norm.weight, norm.variance_epsilon, out_index=om)
            last = i + 1 == len(layers)
            norm = self.model.model.norm if last else layers[i + 1].input_layernorm
            oq = None if last else order_of(layers[i + 1].self_attn)
            y = layer.mlp(x, ordered=True) if om is not None else layer.mlp(x)
            h, x = add_rms_norm(h, y, norm.weight, norm.variance_epsilon, out_index=oq)
        return end(None, None, norm, x)

    def _layers_norm_in_matmul(self, h, position_ids, kv_offset, attend, end):
        """The same stack for a handful of rows: the QKV and the gate/up launch each do the residual
        add and the RMSNorm of their own input (same bits as _layers' separate launches), so a
        layer is 5 launches instead of 7."""
        layers = self.model.model.layers
        h = h.contiguous()  # (the projections that normalise their own input take no strides)
        delta = None
        for layer, (kc, vc) in zip(layers, self.caches):
            attn, n1, n2 = layer.self_attn, layer.input_layernorm, layer.post_attention_layernorm
            q, _, _, h = attn.project_qkv(h, position_ids, kv_out=(kc, vc), kv_offset=kv_offset,
                                          norm=(delta, norm_weight(n1), n1.variance_epsilon))
            h, delta = layer.mlp.forward_normed(h, attn.project_out(*attend(q, kc, vc, attn)), norm_weight(n2), n2.variance_epsilon)
        return end(h, delta, self.model.model.norm, None)

    def _last_tokens(self, h, delta, norm, x):
        """Greedy tokens behind the last position [B, 1]."""
        if x is None:
            _, x = add_rms_norm(h, delta, norm.weight, norm.variance_epsilon)
        return lm_head_argmax(x[:, -1:, :], self.model.lm_head.weight)

    def _end_step(self, h, delta, norm, x):
        """The end of a decode step: tokens and position move on, in place."""
        model = self.model
        if not self.one_launch_end:
            self.tokens.copy_(self._last_tokens(h, delta, norm, x))
            self.position.add_(1)
            return
        w = norm_weight(norm)
        if x is None and self.bsz == 1 and w.numel() <= NORM_MAX_HIDDEN:
            x = h  # (the launch normalises its row itself)
        else:
            if x is None:
                _, x = add_rms_norm(h, delta, w, norm.variance_epsilon)
            delta = w = None
        greedy_step_end(x, delta, w, norm.variance_epsilon, model.lm_head.weight, self.tokens, self.position, self.history)

    @torch.no_grad()
    def prefill(self, input_ids: torch.Tensor) -> torch.Tensor:
        """Run the prompt (positions 0..S-1), fill the caches, return the first new token [B, 1]."""
        bsz, prompt = input_ids.shape
        if bsz != self.bsz or prompt >= self.capacity:
            raise ValueError("prompt does not fit this decoder's batch size / capacity")
        dev = input_ids.device
        position_ids = torch.arange(prompt, device=dev, dtype=torch.int32).unsqueeze(0).expand(bsz, prompt).contiguous()
        def attend(q, kc, vc, attn):
            # the prompt's K and V are in cache rows 0 .. prompt - 1 already; the result comes in o_proj's input layout
            return prefill_attention(q, kc, vc, 0), False

        nxt = self._layers(self.model.model.embed_tokens(input_ids), position_ids, 0, attend, self._last_tokens)
        self.tokens.copy_(nxt)
        self.position.fill_(prompt)
        return nxt

    def _step(self):
        """One decode token from the static buffers: reads tokens and position, writes them back."""

        def attend(q, kc, vc, attn):  # rows 0..position of the cache; act-order o_proj: written in the order it reads
            order = attn.context_order()
            return decode_attention(q, kc, vc, self.position, out_index=order), order is not None

        self._layers(self.model.model.embed_tokens(self.tokens), self.position, KV_AT_POSITION, attend, self._end_step)

    @torch.no_grad()
    def decode(self, steps: int, use_graph: bool = False) -> torch.Tensor:
        """`steps` more greedy tokens after prefill -> [B, steps]."""
        if steps < 0:
            raise RuntimeError(f"decode of {steps} steps")
        # where the sequences stand is read back: the kernels move `position` on, also in a step that is interrupted on the host
        # and in a replay of `graph` by the caller, and the caller may write to it
        stand = self.position.flatten().tolist()
        if max(stand) + steps > self.capacity:
            raise ValueError("decode would run past the cache capacity")
        if use_graph and self.graph is None and steps > 0:
            self._capture()
        # the tokens are at their places in `history` afterwards; where the sequences stand at different places, or the step
        # does not keep them there, they are collected one by one
        at = stand[0]
        kept = (self._graph_keeps_history if use_graph else self.one_launch_end) and at >= 0 and min(stand) == max(stand)
        out = None if kept else torch.empty((self.bsz, steps), dtype=torch.long, device=self.tokens.device)
        for i in range(steps):
            if use_graph:
                self.graph.replay()
            else:
                self._step()
            if not kept:
                out[:, i:i + 1].copy_(self.tokens)
        if kept:
            out = self.history[:, at + 1:at + 1 + steps].clone()
        # one 4-byte read per workspace: a bounded wait of the small-M kernels that ran out would have made tokens wrong silently
        _lib.check_exchange_errors()
        return out

    def _capture(self):
        """Capture _step as a graph.  The warm-up steps run on the capture stream first, so
        workspaces and tables exist before capture; their effect on tokens, position and the
        cache rows they wrote is undone (the rows lie beyond the current position and are
        rewritten before any later step attends to them)."""
        tokens0, position0 = self.tokens.clone(), self.position.clone()
        side = torch.cuda.Stream(device=self.tokens.device)
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            self._step()
            self.tokens.copy_(tokens0)
            self.position.copy_(position0)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        self._graph_keeps_history = self.one_launch_end
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph, stream=side):
            self._step()
        self.tokens.copy_(tokens0)
        self.position.copy_(position0)
        torch.cuda.synchronize()
