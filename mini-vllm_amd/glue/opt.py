"""OPT decoder glue (mirror of minivllm/models/opt.py): learned positions (offset 2), MHA,
LayerNorm, ReLU MLP, pre- or post-LN.  Attention runs on the same HIP kernels (D = 64 for
OPT-125M); LayerNorm/ReLU/bias adds stay torch ops — OPT is the reference's CPU plumbing
config, not a throughput target — but in fp32 prompts, where they ride in the projections (csrc/linear_f32.hip)."""
from __future__ import annotations

from typing import Any

import torch
import torch.nn.functional as F
from torch import nn
from torch.nn.modules import module as _modules

from .. import hip_ops
from ..layers import (Attention, ColumnParallelLinear, ParallelLMHead, QKVParallelLinear, RowParallelLinear,
                      VocabParallelEmbedding)
from ..layers.linear import f32_tiles
from ..parallel_state import get_tensor_parallel_world_size

__all__ = ["OPTForCausalLM"]

# fp32 layers go by parts of bf16 as a whole (norms, ReLU and residual sums within the projections' launches) from so many tiles of 64 x 64 hidden features
# and so many rows on, which have to pay for the weights' parts whatever the width.  us, projections and what is between them, as modules / as a whole:
# 768 features: 1025 rows (204 tiles) 173 / 174, 1300 (252) 181 / 184, 1345 (264) 194 / 203, 1408 (264) 205 / 203, 1600 (300) 215 / 205, 1664 247 / 210; 1024: 769 (208) 200 / 222,
# 1088 (272) 261 / 260, 1345 316 / 282; 2048: 513 (288) 474 / 562, 769 600 / 617, 1025 813 / 772; 4096: 257 (320) 933 / 1432, 513 1660 / 1733, 769 2238 / 2208,
# 1025 2811 / 2795; 5120: 257 1640 / 1967, 1025 4532 / 4464; 7168: 129 (336) 1567 / 2979, 513 5278 / 5267, 1025 7296 / 7398
F32_LAYER_TILES_MIN, F32_LAYER_ROWS_MIN = 264, 1024


class OPTLearnedPositionalEmbedding(nn.Embedding):
    def __init__(self, num_embeddings: int, embedding_dim: int):
        self.offset = 2
        super().__init__(num_embeddings + self.offset, embedding_dim)

    def forward(self, positions):
        return super().forward(positions + self.offset)


class OPTAttention(nn.Module):
    def __init__(self, embed_dim: int, num_heads: int, bias: bool = True) -> None:
        super().__init__()
        if embed_dim % num_heads:
            raise ValueError(f"embed_dim must be divisible by num_heads (got 'embed_dim': {embed_dim} "
                             f"and 'num_heads': {num_heads}).")
        tp = get_tensor_parallel_world_size()
        self.embed_dim, self.total_num_heads = embed_dim, num_heads
        self.num_heads = num_heads // tp
        self.head_dim = embed_dim // num_heads
        self.scaling = self.head_dim ** -0.5
        self.qkv_proj = QKVParallelLinear(embed_dim, self.head_dim, num_heads, bias=bias)
        self.out_proj = RowParallelLinear(embed_dim, embed_dim, bias=bias)
        self.attn = Attention(self.num_heads, self.head_dim, self.scaling, self.num_heads)

    def forward(self, positions, hidden_states):
        return self.out_proj(self.attend(self.qkv_proj(hidden_states)))

    def attend(self, qkv):
        t = qkv.shape[0]
        width = self.num_heads * self.head_dim
        q, k, v = (qkv[:, i * width:(i + 1) * width].view(t, self.num_heads, self.head_dim) for i in range(3))
        o = self.attn(q, k, v)  # stores K/V, then prefill / paged decode
        return o.reshape(t, width)


class OPTDecoderLayer(nn.Module):
    def __init__(self, config) -> None:
        super().__init__()
        d = config.hidden_size
        self.self_attn = OPTAttention(d, config.num_attention_heads, bias=config.enable_bias)
        self.do_layer_norm_before = config.do_layer_norm_before
        self.self_attn_layer_norm = nn.LayerNorm(d)
        self.fc1 = ColumnParallelLinear(d, config.ffn_dim, bias=config.enable_bias)
        self.fc2 = RowParallelLinear(config.ffn_dim, d, bias=config.enable_bias)
        self.final_layer_norm = nn.LayerNorm(d)
        self.parts_rows = max(F32_LAYER_ROWS_MIN, (-(-F32_LAYER_TILES_MIN // -(-d // 64)) - 1) * 64 + 1)   # the fewest rows

    def _by_parts(self, x) -> bool:
        if x.shape[0] < self.parts_rows or x.dtype != torch.float32:   # (small steps are bound by the host: nothing else is looked at)
            return False
        att = self.self_attn
        if not self.do_layer_norm_before or f32_tiles(x.shape[0], x.shape[1]) < F32_LAYER_TILES_MIN or type(att) is not OPTAttention:
            return False
        # modules that are not called: nobody may have put another in their place, or wait for a call
        linears, norms = (att.qkv_proj, att.out_proj, self.fc1, self.fc2), (self.self_attn_layer_norm, self.final_layer_norm)
        if tuple(map(type, linears)) != (QKVParallelLinear, RowParallelLinear, ColumnParallelLinear, RowParallelLinear) \
                or any(type(norm) is not nn.LayerNorm or norm.weight is None or norm.normalized_shape != (x.shape[1],) for norm in norms):
            return False
        if _modules._global_forward_hooks or _modules._global_forward_pre_hooks \
                or any(m._forward_hooks or m._forward_pre_hooks or "forward" in m.__dict__ for m in (*linears, *norms, att)):
            return False
        return all(lin.tp_size == 1 for lin in linears) and hip_ops.linear_f32_ok(x, *(t for m in (*linears, *norms) for t in (m.weight, m.bias)))

    def _forward_parts(self, x):
        att, fc1, fc2 = self.self_attn, self.fc1, self.fc2
        rows, w_qkv, w_out = hip_ops.split_f32(x, att.qkv_proj.weight, att.out_proj.weight, norm=self.self_attn_layer_norm)
        rows, = hip_ops.split_f32(att.attend(hip_ops.linear_f32(rows, w_qkv, att.qkv_proj.bias)))
        x = hip_ops.linear_f32(rows, w_out, att.out_proj.bias, residual=x)
        rows, w1, w2 = hip_ops.split_f32(x, fc1.weight, fc2.weight, norm=self.final_layer_norm)
        return hip_ops.linear_f32(hip_ops.linear_f32(rows, w1, fc1.bias, relu=True, parts=True), w2, fc2.bias, residual=x)

    def forward(self, positions, x, residual=None):
        if self._by_parts(x):
            return self._forward_parts(x), None
        if self.do_layer_norm_before:
            x = x + self.self_attn(positions, self.self_attn_layer_norm(x))
            x = x + self.fc2(F.relu(self.fc1(self.final_layer_norm(x))))
        else:
            x = self.self_attn_layer_norm(x + self.self_attn(positions, x))
            x = self.final_layer_norm(x + self.fc2(F.relu(self.fc1(x))))
        return x, None


class OPTDecoder(nn.Module):
    def __init__(self, config) -> None:
        super().__init__()
        self.config = config
        d, w = config.hidden_size, config.word_embed_proj_dim
        self.embed_tokens = VocabParallelEmbedding(config.vocab_size, d)
        self.embed_positions = OPTLearnedPositionalEmbedding(config.max_position_embeddings, d)
        self.project_in = nn.Linear(w, d, bias=False) if w != d else None
        self.project_out = nn.Linear(d, w, bias=False) if w != d else None
        self.final_layer_norm = nn.LayerNorm(d) if config.do_layer_norm_before else None
        self.layers = nn.ModuleList(OPTDecoderLayer(config) for _ in range(config.num_hidden_layers))

    def forward(self, input_ids, positions):
        x = self.embed_tokens(input_ids)
        if self.project_in is not None:
            x = self.project_in(x)
        x = x + self.embed_positions(positions)
        for layer in self.layers:
            x, _ = layer(positions, x, None)
        if self.final_layer_norm is not None:
            x = self.final_layer_norm(x)
        if self.project_out is not None:
            x = self.project_out(x)
        return x


class OPTModel(nn.Module):
    def __init__(self, config) -> None:
        super().__init__()
        self.decoder = OPTDecoder(config)

    def forward(self, input_ids, positions):
        return self.decoder(input_ids, positions)


class OPTForCausalLM(nn.Module):
    packed_modules_mapping = {"q_proj": ("qkv_proj", "q"), "k_proj": ("qkv_proj", "k"), "v_proj": ("qkv_proj", "v")}

    def __init__(self, config) -> None:
        super().__init__()
        self.config = config
        self.model = OPTModel(config)
        self.lm_head = ParallelLMHead(config.vocab_size, config.hidden_size)
        if config.tie_word_embeddings:
            self.lm_head.weight = self.model.decoder.embed_tokens.weight

    def forward(self, input_ids, positions):
        return self.model(input_ids, positions)

    def compute_logits(self, hidden_states, gather: bool = True):
        return self.lm_head(hidden_states, gather=gather)

    def set_kv_cache(self, kv_cache) -> None:
        for layer, (k, v) in zip(self.model.decoder.layers, kv_cache):
            layer.self_attn.attn.k_cache, layer.self_attn.attn.v_cache = k, v

    def load_weights(self, weights: dict[str, Any]) -> None:
        from ..utils.loader import load_weight

        for name, tensor in weights.items():
            load_weight(self, name, tensor, self.packed_modules_mapping)
