"""Gated-DeltaNet / softmax hybrid token mixer with the forward signature, returns and parameter
names of the reference layer (src/nats/layers/natsl_attn_gdn.py:64-666).

Projections, short convolutions and norms are torch; block pooling, the selector, the mixed operator
and the output norm-gate are the HIP kernels of this package.  Training works, with HIP backwards throughout: the softmax
branch (natsl_softmax_sparse_bwd), the linear branch (natsl_linear_chunk_bwd), the short convolutions
(natsl_short_conv_bwd), the row norms (natsl_row_norm_bwd) and the norm-gate (natsl_norm_gate_bwd); only the block pooling's
backward (a broadcast of the block's gradient) and the projections are torch operations.  With a NAtSCache
the layer prefills in chunk mode and decodes in steps of fewer than 64 tokens; 64 or more new tokens on a cache that already
holds tokens (a second prompt) run through the chunked operators again, the linear branch from the state that entered the
incomplete block and the softmax branch with the kept blocks as a key prefix (the reference's attention operator cannot run
this case: it sizes its output by the keys, src/nats/ops/attns/attns.py:1439,1491).
"""
from __future__ import annotations

import math
from typing import Optional

import torch
import torch.nn as nn
import torch.nn.functional as F

from . import nats_util
from ._front import fast_front
from ._layer_step import layer_step
from ._mixed_common import state_behind
from .cache import NAtSCache, NAtSLayerCache
from .mixed_attn_gdn import nats_mixed_attn_gdn, nats_mixed_attn_gdn_chunk_inference, nats_mixed_attn_gdn_recurrent
from .modules import FusedMultiInputRMSNormGated, RMSNorm, ShortConvolution


class NeuralAttentionSearchLinearAttnGDN(nn.Module):
    def __init__(self, hidden_size: int = 2048, expand_v: float = 2, head_dim: int = 256, num_heads: int = 6,
                 num_attn_heads: int = 24, num_v_heads: int = None, n_ops: int = 2, num_nats_head: Optional[int] = None,
                 nats_block_size: int = 64, nats_block_agg_type: str = 'mean', nats_sample_strategy: str = 'argmax',
                 ops_for_incomplete_chunks: str = 'all', mode: str = 'chunk', use_gate: bool = True,
                 use_short_conv: bool = True, allow_neg_eigval: bool = False, conv_size: int = 4, conv_bias: bool = False,
                 conv_activation: Optional[str] = 'silu', outputs_are_weighted: bool = True, attn_qk_norm: bool = True,
                 attn_with_short_conv: bool = True, compute_dnats_for_invalid_blocks_attn: bool = False,
                 compute_dnats_for_invalid_blocks_linear_att: bool = False, decay_for_non_gdn_blocks: bool = True,
                 incomplete_block_start_with_ht: bool = True, attn_apply_pos_encoding: bool = False,
                 attn_rope_theta: Optional[float] = 10000., attn_max_position_embeddings: Optional[int] = None,
                 layer_idx: int = None, norm_eps: float = 1e-5, **kwargs):
        super().__init__()
        if n_ops != 2:
            raise NotImplementedError("two ops (softmax, linear) are built")
        if nats_block_agg_type != 'mean':
            raise NotImplementedError(f"Pooling system {nats_block_agg_type} is not supported!")
        if nats_sample_strategy != 'argmax':
            raise NotImplementedError("only the hard (argmax) selector is built")
        if attn_apply_pos_encoding:
            raise NotImplementedError("rotary position encoding for the attention view is not built")
        if not use_gate or not outputs_are_weighted:
            raise NotImplementedError("only use_gate=True with weighted outputs (the published configuration) is built")
        assert mode in ['chunk', 'fused_recurrent'], f"Not supported mode `{mode}`."
        self.mode, self.hidden_size, self.expand_v = mode, hidden_size, expand_v
        self.allow_neg_eigval, self.use_gate, self.use_short_conv = allow_neg_eigval, use_gate, use_short_conv
        self.conv_size, self.conv_bias = conv_size, conv_bias
        self.head_dim, self.num_heads = head_dim, num_heads
        self.num_v_heads = num_v_heads if num_v_heads is not None else num_heads
        self.n_ops = n_ops
        self.head_k_dim = head_dim
        self.head_v_dim = int(head_dim * expand_v)
        self.key_dim = int(num_heads * self.head_k_dim)
        self.value_dim = int(self.num_v_heads * self.head_v_dim)
        self.layer_idx = layer_idx
        self.attn_qk_norm, self.num_attn_heads = attn_qk_norm, num_attn_heads
        self.head_attn_k_dim = self.key_dim // num_attn_heads
        self.head_attn_v_dim = self.value_dim // num_attn_heads
        self.attn_with_short_conv = attn_with_short_conv
        self.incomplete_block_start_with_ht = incomplete_block_start_with_ht
        self.decay_for_non_gdn_blocks = decay_for_non_gdn_blocks
        self.compute_dnats_for_invalid_blocks_attn = compute_dnats_for_invalid_blocks_attn
        self.compute_dnats_for_invalid_blocks_linear_att = compute_dnats_for_invalid_blocks_linear_att
        self.nats_block_size = nats_block_size
        self.num_nats_head = num_heads if num_nats_head is None else num_nats_head
        self.ops_for_incomplete_chunks = ops_for_incomplete_chunks
        self.outputs_are_weighted = outputs_are_weighted
        if not math.isclose(self.num_v_heads * head_dim * expand_v, self.value_dim, rel_tol=1e-5):
            raise ValueError(f"expand_v={expand_v} does not produce an integer value_dim")
        if self.num_v_heads > num_heads and self.num_v_heads % num_heads != 0:
            raise ValueError(f"num_v_heads={self.num_v_heads} must be divisible by num_heads={num_heads}.")
        if num_attn_heads > num_heads and num_attn_heads % num_heads != 0:
            raise ValueError(f"num_attn_heads={num_attn_heads} must be divisible by num_heads={num_heads}.")

        if attn_qk_norm:
            self.q_norm = RMSNorm(self.head_attn_k_dim, eps=norm_eps)
            self.k_norm = RMSNorm(self.head_attn_k_dim, eps=norm_eps)
        self.q_proj = nn.Linear(hidden_size, self.key_dim, bias=False)
        self.k_proj = nn.Linear(hidden_size, self.key_dim, bias=False)
        self.v_proj = nn.Linear(hidden_size, self.value_dim, bias=False)
        self.a_proj = nn.Linear(hidden_size, self.num_v_heads, bias=False)
        self.b_proj = nn.Linear(hidden_size, self.num_v_heads, bias=False)
        self.nats_layer = nn.Linear(hidden_size, n_ops * self.num_nats_head, bias=False)
        A = torch.empty(self.num_v_heads, dtype=torch.float32).uniform_(0, 16)
        self.A_log = nn.Parameter(torch.log(A))
        dt = torch.exp(torch.rand(self.num_v_heads) * (math.log(0.1) - math.log(0.001)) + math.log(0.001)).clamp(min=1e-4)
        self.dt_bias = nn.Parameter(dt + torch.log(-torch.expm1(-dt)))
        self.nats_out_weights_layer = nn.Linear(self.key_dim, n_ops * num_attn_heads, bias=False)
        if use_short_conv:
            self.q_conv1d = ShortConvolution(self.key_dim, conv_size, conv_bias, conv_activation)
            self.k_conv1d = ShortConvolution(self.key_dim, conv_size, conv_bias, conv_activation)
            self.v_conv1d = ShortConvolution(self.value_dim, conv_size, conv_bias, conv_activation)
        self.g_proj = nn.Linear(hidden_size, self.value_dim, bias=False)
        self.o_norm = FusedMultiInputRMSNormGated(self.head_attn_v_dim, eps=norm_eps)
        self.o_proj = nn.Linear(self.value_dim, hidden_size, bias=False)
        self.attn_fraction = torch.zeros(1)

    # -- pieces of the forward, also used by the parity test ---------------------------------------
    def select_ops(self, hidden_states: torch.Tensor, cu_seqlens=None, force_last_block: bool = True):
        """Selector: block means -> nats_layer -> hard selection, with the last block forced to both ops unless
        told otherwise (reference :411-420, :553-555, :579-583).  Returns (types [B,TN,HN,2], n_nats_blocks int32
        [B,HN,2], the last block's type before forcing [B,HN,2])."""
        B, _, dim = hidden_states.shape
        pooled = nats_util.mean_pooling(hidden_states.unsqueeze(-2), self.nats_block_size, cu_seqlens=cu_seqlens)
        pooled = pooled.view(B, pooled.shape[1], dim)
        logits = self.nats_layer(pooled).unflatten(-1, (self.num_nats_head, self.n_ops))
        types, n_blocks = nats_util.hard_select(logits, force_last_block=False)
        last = types[:, -1].clone()
        if force_last_block:
            n_blocks = n_blocks + (1 - last.to(torch.int32))      # counts after forcing the last block to 1
            types[:, -1] = 1
        return types, n_blocks, last

    def _layer_cache(self, past_key_values) -> Optional[NAtSLayerCache]:
        """The layer's own cache, created on first use (reference :391-402)."""
        if past_key_values is None:
            return None
        if self.layer_idx is None:
            raise ValueError("a layer that uses a cache needs its layer_idx")
        while len(past_key_values) <= self.layer_idx:
            past_key_values.add_natsl_layer_cache(0, n_tokens_in_nats_block=0, n_attn_blocks=None,
                                                  nats_block_size=self.nats_block_size,
                                                  op_for_incomplete_chunk=self.ops_for_incomplete_chunks)
        return past_key_values[self.layer_idx]

    def _general_front(self, hidden_states, selector_input, conv_states, use_cache, cu_seqlens):
        """Selector, projections, convolutions, norms and gates through the submodules one by one."""
        if selector_input is not None:
            raw_types, _, _ = self.select_ops(selector_input, cu_seqlens, force_last_block=False)
        else:
            raw_types = torch.ones(hidden_states.shape[0], 1, self.num_nats_head, self.n_ops, device=hidden_states.device, dtype=hidden_states.dtype)

        new_conv_states = []

        def conv_or_act(x, conv, state):
            if self.use_short_conv:
                y, final = conv(x=x, cache=state, output_final_state=bool(use_cache), cu_seqlens=cu_seqlens)
                new_conv_states.append(final)
                return y
            return F.silu(x)

        if self.attn_with_short_conv:
            q = conv_or_act(self.q_proj(hidden_states), getattr(self, 'q_conv1d', None), conv_states[0])
            k = conv_or_act(self.k_proj(hidden_states), getattr(self, 'k_conv1d', None), conv_states[1])
            v = conv_or_act(self.v_proj(hidden_states), getattr(self, 'v_conv1d', None), conv_states[2])
            q_attn, k_attn, v_attn = q, k, v
        else:
            q_attn, k_attn, v_attn = self.q_proj(hidden_states), self.k_proj(hidden_states), self.v_proj(hidden_states)
            q = conv_or_act(q_attn, getattr(self, 'q_conv1d', None), conv_states[0])
            k = conv_or_act(k_attn, getattr(self, 'k_conv1d', None), conv_states[1])
            v = conv_or_act(v_attn, getattr(self, 'v_conv1d', None), conv_states[2])
        o_weights = self.nats_out_weights_layer(q).unflatten(-1, (self.num_attn_heads, self.n_ops)).softmax(-1)

        q, k = (x.unflatten(-1, (-1, self.head_k_dim)) for x in (q, k))
        v = v.unflatten(-1, (-1, self.head_v_dim))
        q_attn, k_attn = (x.unflatten(-1, (-1, self.head_attn_k_dim)) for x in (q_attn, k_attn))
        v_attn = v_attn.unflatten(-1, (-1, self.head_attn_v_dim))
        if self.num_v_heads > self.num_heads:
            q, k = (x.repeat_interleave(self.num_v_heads // self.num_heads, dim=-2) for x in (q, k))
        if self.attn_qk_norm:
            q_attn, k_attn = self.q_norm(q_attn), self.k_norm(k_attn)

        beta = self.b_proj(hidden_states).sigmoid()
        if self.allow_neg_eigval:
            beta = beta * 2.
        g = -self.A_log.float().exp() * F.softplus(self.a_proj(hidden_states).float() + self.dt_bias)
        return q, k, v, q_attn, k_attn, v_attn, o_weights, g, beta, raw_types, tuple(new_conv_states) if self.use_short_conv else None

    def _into_cache(self, cache, q_len, raw_types, attn_kv, lattn, conv_states, state, state_entering, g_sum):
        """An empty cache after its first prompt (FastFront.prompt's outputs)."""
        k, v, beta, g = lattn
        cache.update_attn_cache(attn_kv, nats_block_types=raw_types)
        cache.update_lattn_cache((k, v), beta, g, 'chunk', self.ops_for_incomplete_chunks)
        if q_len % self.nats_block_size == 0:
            state_entering = state_behind(state, state_entering, g_sum if self.decay_for_non_gdn_blocks else None, raw_types[:, -1])
        self.last_recurrent_state, self.last_block_start_state = state, state_entering
        cache.update(recurrent_state=state, recurrent_state_block_start=state_entering, attn_state=attn_kv, conv_state=conv_states,
                     nats_block_types=raw_types, l_attn_state=(k, v), g=g, n_new_tokens=q_len)

    def forward(self, hidden_states: torch.Tensor, attention_mask: Optional[torch.Tensor] = None, past_key_values=None,
                use_cache: Optional[bool] = False, output_attentions: Optional[bool] = False, **kwargs):
        if attention_mask is not None:
            assert len(attention_mask.shape) == 2, "Expected attention_mask as a 0-1 matrix with shape [batch_size, seq_len]"
            if len(attention_mask) > 1:
                raise NotImplementedError("Attention with variable length is not supported yet!")
        B, q_len, _ = hidden_states.shape
        mode = 'fused_recurrent' if q_len < 64 else self.mode                  # reference :387
        if self.training:
            assert mode == 'chunk', "Only chunk mode is supported in training."
        cu_seqlens = kwargs.get('cu_seqlens', None)
        cache = self._layer_cache(past_key_values)
        if cache is None and mode != 'chunk':
            raise ValueError("fewer than 64 tokens are decoded on a cache: pass past_key_values")
        # 64 or more new tokens on a cache that already holds tokens (a second prompt): the chunked operators run again, the
        # linear branch from the state that entered the incomplete block (its cached tokens in front of the new ones), the
        # softmax branch with the kept blocks as a key prefix
        continuing = cache is not None and mode == 'chunk' and cache.n_observed_tokens > 0
        if cache is not None and cu_seqlens is not None:
            raise NotImplementedError("packed sequences are not supported together with a cache")

        if cache is not None and mode != 'chunk' and q_len > 1:
            if cache._n_tokens_in_nats_block + q_len > self.nats_block_size:
                # the step crosses a selector-block boundary: the tokens that complete the block first (the block gets its
                # type and the cache is updated), then the rest as the start of the next block -- what the reference's
                # recurrent kernel does with two blocks in one call (src/nats/ops/gated_delta_rule/fused_recurrent.py:144-358)
                first = self.nats_block_size - cache._n_tokens_in_nats_block
                kw = dict(past_key_values=past_key_values, use_cache=use_cache, output_attentions=output_attentions, **kwargs)
                o1 = self.forward(hidden_states[:, :first], attention_mask, **kw)[0]
                o2 = self.forward(hidden_states[:, first:], attention_mask, **kw)[0]
                return torch.cat([o1, o2], 1), None, past_key_values
        if cache is not None and mode != 'chunk' and use_cache:
            o = layer_step(self, 'gdn', hidden_states, cache)
            if o is not None:
                return o, None, past_key_values
        # selector: on a cache, over the tokens of the incomplete block + the new ones, once they complete a block
        if cache is not None:
            selector_input = cache.update_attn_types(input_hidden_states=hidden_states)
        else:
            selector_input = hidden_states
        fast = None
        if mode == 'chunk' and selector_input is not None and getattr(self.select_ops, '__func__', None) is _SELECT_OPS:
            fast = fast_front(self, 'gdn', hidden_states, cache, cu_seqlens)
        if fast is not None and fast.native is not None and (not use_cache if cache is None else use_cache and cache.is_empty()) and \
                (nats_mixed_attn_gdn, nats_mixed_attn_gdn_chunk_inference) == _OPERATORS:
            if self.training and cache is None:
                o, self.attn_fraction = fast.train(hidden_states)
                self.last_recurrent_state = self.last_block_start_state = None
                return o, None, past_key_values
            if not self.training and not fast.grad(hidden_states, *fast.w.values(), fast.wn):
                o, self.attn_fraction, kept = fast.prompt(hidden_states, None if cache is None else lambda types: cache.foresee(types, q_len))
                self.last_recurrent_state = self.last_block_start_state = None
                if cache is not None:
                    self._into_cache(cache, q_len, *kept)
                return o, None, past_key_values
        types = n_nats_blocks = None
        conv_states = cache.conv_state if cache is not None and cache.conv_state is not None else (None, None, None)
        if fast is not None:
            whole = selector_input is hidden_states
            q, k, v, gate, (g, beta, _), logits = fast.project(hidden_states, self.nats_block_size if whole else 0, self.nats_layer)
            if not whole:
                logits = self.nats_layer(nats_util.mean_pooling(selector_input, self.nats_block_size))
            logits = logits.unflatten(-1, (self.num_nats_head, self.n_ops))
            # (the types before the last block is forced are only needed where states are handed on)
            types, n_nats_blocks, attn_fraction, raw_types = fast.select(logits, bool(use_cache) or cache is not None)
            if cache is not None:
                cache.foresee(raw_types, q_len)
            q, k, v, q_attn, k_attn, o_mix, _, _, v_attn, new_conv_states = fast.conv_norm(q, k, v, conv_states, bool(use_cache))
            q, k = (x.unflatten(-1, (-1, self.head_k_dim)) for x in (q, k))
            v = v.unflatten(-1, (-1, self.head_v_dim))
            q_attn, k_attn = (x.unflatten(-1, (-1, self.head_attn_k_dim)) for x in (q_attn, k_attn))
            v_attn = v_attn.unflatten(-1, (-1, self.head_attn_v_dim))
        else:
            q, k, v, q_attn, k_attn, v_attn, o_mix, g, beta, raw_types, new_conv_states = self._general_front(
                hidden_states, selector_input, conv_states, use_cache, cu_seqlens)
            gate = None

        state, state_block_start, g_cumsum = None, None, None
        k_new, v_new, g_new = k_attn, v_attn, g
        if cache is not None:
            k_attn, v_attn = cache.update_attn_cache((k_attn, v_attn), nats_block_types=raw_types)
            k, v, beta, g = cache.update_lattn_cache((k, v), beta, g, mode, self.ops_for_incomplete_chunks)
            state, state_block_start, g_cumsum = cache.recurrent_state, cache.recurrent_state_block_start, cache.g_cumsum
        n_cached, prefix_valid = 0, None
        if continuing:
            # keys: the kept blocks, the incomplete block's cached tokens, the new tokens -- the cache's buffer as it lies; the
            # linear inputs came back with the incomplete block's tokens in front; the queries of those tokens are not needed
            n_cached = cache._n_tokens_in_nats_block
            n_keys = cache.n_attn_tokens_max + q_len
            k_attn, v_attn = cache.attn_k[:, :n_keys], cache.attn_v[:, :n_keys]
            if cache.n_attn_blocks_max > 0:
                prefix_valid = cache.valid_attn_tokens[:, :cache.n_attn_blocks_max]
            if n_cached:
                front = lambda t: torch.cat([t.new_zeros(t.shape[0], n_cached, *t.shape[2:]), t], 1)
                q, q_attn = front(q), front(q_attn)
                state = state_block_start

        common = dict(q_attn=q_attn, k_attn=k_attn, v_attn=v_attn, q_lattn=q, k_lattn=k, v_lattn=v, g=g, beta=beta,
                      scale_attn=k_attn.shape[-1] ** -0.5, scale_lattn=k.shape[-1] ** -0.5, cu_seqlens=cu_seqlens,
                      cu_seqlens_nats=None, nats_block_size=self.nats_block_size,
                      ops_for_incomplete_chunks=self.ops_for_incomplete_chunks,
                      output_final_state_gated_delta=bool(use_cache),
                      incomplete_block_start_with_ht=self.incomplete_block_start_with_ht,
                      decay_for_non_gdn_blocks=self.decay_for_non_gdn_blocks, use_g_for_attn=False,
                      lattn_use_qk_l2norm_in_kernel=True)
        if mode == 'chunk':
            # the last block runs both ops so that its state is recorded (reference :547-555, :577-583)
            last_type = raw_types[:, -1].clone() if types is None else raw_types[:, -1]
            if types is None:
                types = raw_types.clone()
                types[:, -1] = 1
                n_nats_blocks = types.to(torch.int32).sum(1)
            self.attn_fraction = attn_fraction if fast is not None else n_nats_blocks[..., 0].sum(0).float() / (types.shape[1] * B)
            if self.training:
                o_lin, o_attn, state = nats_mixed_attn_gdn(
                    initial_state_gated_delta=state, nats_block_types=types, n_nats_blocks=n_nats_blocks,
                    compute_dnats_for_invalid_blocks_attn=self.compute_dnats_for_invalid_blocks_attn,
                    compute_dnats_for_invalid_blocks_linear_att=self.compute_dnats_for_invalid_blocks_linear_att, **common)
                state_block_start = None
            else:
                o_lin, o_attn, state, state_block_start = nats_mixed_attn_gdn_chunk_inference(
                    initial_state_gated_delta_chunk_start=state if continuing else state_block_start, nats_block_types=types,
                    n_nats_blocks=n_nats_blocks, attn_prefix_valid=prefix_valid,
                    op_type_last_chunk=last_type if k.shape[1] % self.nats_block_size == 0 else None, **common)
                o_lin, o_attn = o_lin[:, n_cached:], o_attn[:, n_cached:]
        else:
            attn_msk = cache.generate_msk(n_data=q_len, nats_block_types=raw_types,
                                          compute_incomplete_chunk=self.ops_for_incomplete_chunks != 'gated_delta_net')
            o_lin, o_attn, state, state_block_start = nats_mixed_attn_gdn_recurrent(
                attn_msk=attn_msk, initial_state_gated_delta=state, initial_state_gated_delta_chunk_start=state_block_start,
                g_cumsum=g_cumsum, nats_block_types=raw_types, n_tokens_in_current_block=cache._n_tokens_in_nats_block, **common)
        self.last_recurrent_state, self.last_block_start_state = state, state_block_start

        if cache is not None:
            cache.update(recurrent_state=state, recurrent_state_block_start=state_block_start, attn_state=(k_new, v_new),
                         conv_state=new_conv_states, nats_block_types=raw_types,
                         l_attn_state=(k, v), g=g_new, n_new_tokens=q_len)

        if fast is not None:
            return fast.tail(o_lin.reshape(o_attn.shape), o_attn, gate.view(o_attn.shape), o_mix), None, past_key_values
        gate = self.g_proj(hidden_states).unflatten(-1, (-1, self.head_v_dim))
        o = self.o_norm(o_lin.reshape(o_attn.shape), o_attn, gate.reshape(o_attn.shape), o_mix)
        o = self.o_proj(o.flatten(-2))
        return o, None, past_key_values


# the selector that the fused front contains; a layer whose select_ops is another one takes the general front, which calls it
_SELECT_OPS = NeuralAttentionSearchLinearAttnGDN.select_ops
# ... and the operators: where others stand in their places, those are called
_OPERATORS = (nats_mixed_attn_gdn, nats_mixed_attn_gdn_chunk_inference)
