"""Llama-family decoder (Llama-3 8B / 70B architectures) for the MI355X
engine.

Compute path (SURVEY.md §7 stage 3): GEMMs via ops.linear (hipBLASLt on ROCm,
TP-sharded through parallel.layers); everything between them is a
hand-written gfx950 kernel — fused add+RMSNorm, NeoX RoPE, paged-cache
append, MFMA flash prefill / paged decode attention, fused SwiGLU. On CPU
the ops package transparently runs the fp32 references so the same module
is testable without a GPU.
"""
from __future__ import annotations

from typing import List, Tuple

import torch
import torch.nn as nn
import torch.nn.functional as F

from ... import ops
from ...parallel.comm import tp_rank, tp_world_size
from ...parallel.layers import (ColumnParallelLinear, ReplicatedLinear,
                                RowParallelLinear, _init_weight,
                                calls_plainly)
from ..config import ModelConfig
from .batch import ForwardBatch


# Rows whose products norm for themselves (ops.norm_linear).  Every workgroup does
# so, which from four rows on takes longer than a launch of the norm's own (us, norm
# and product, apart and as one, K = 4096: 1 / 2 / 3 / 4 / 5 rows of 6144 outputs 12.0
# 13.0 14.0 15.0 16.5 and 10.7 12.9 15.0 16.8 19.8, of 28672 as SwiGLU 39.8 40.3 40.5
# 41.2 42.4 and 37.8 39.1 40.5 42.4 47.9; steps of four such layers, 700 tokens each, 3 /
# 4 / 6 sequences 583.9 604.4 650.8 and 582.1 610.8 675.2).  From seven on products may
# come in parts that the norm adds (ops.linear_add_rmsnorm).
FEW_ROWS = 3


def _seed(name: str) -> int:
    # deterministic ACROSS PROCESSES: python's hash() is salted per process,
    # which would give each TP rank different weights (caught by the gloo
    # world_size=2 CPU test)
    import zlib

    return zlib.crc32(name.encode()) & 0x7FFFFFFF


class LlamaAttention(nn.Module):
    def __init__(self, cfg: ModelConfig, layer: int, device, dtype):
        super().__init__()
        tp, rank = tp_world_size(), tp_rank()
        assert cfg.num_heads % tp == 0 and cfg.num_kv_heads % tp == 0, (
            f"TP={tp} must divide heads {cfg.num_heads}/{cfg.num_kv_heads}"
        )
        self.nq = cfg.num_heads // tp
        self.nkv = cfg.num_kv_heads // tp
        self.hd = cfg.head_dim
        self.scale = cfg.head_dim**-0.5
        h = cfg.hidden_size
        # fused qkv: column-parallel over heads (q shard + k shard + v shard)
        q_proj = ColumnParallelLinear(
            h, cfg.num_heads * self.hd, rank, tp, device, dtype,
            _seed(f"l{layer}.q"))
        k_proj = ColumnParallelLinear(
            h, cfg.num_kv_heads * self.hd, rank, tp, device, dtype,
            _seed(f"l{layer}.k"))
        v_proj = ColumnParallelLinear(
            h, cfg.num_kv_heads * self.hd, rank, tp, device, dtype,
            _seed(f"l{layer}.v"))
        # one fused qkv GEMM per layer (decode is launch/skinny-M bound)
        self.qkv = nn.Parameter(
            torch.cat([q_proj.weight.data, k_proj.weight.data,
                       v_proj.weight.data], 0).contiguous(),
            requires_grad=False)
        del q_proj, k_proj, v_proj
        if cfg.qkv_bias:
            # Qwen2 family: bias on qkv only, sharded with the head dims
            # (zeros under synthetic init; real values come from the
            # checkpoint loader)
            self.qkv_b = nn.Parameter(
                torch.zeros((self.nq + 2 * self.nkv) * self.hd,
                            dtype=dtype, device=device),
                requires_grad=False)
        else:
            self.qkv_b = None
        self.o_proj = RowParallelLinear(
            cfg.num_heads * self.hd, h, rank, tp, device, dtype,
            _seed(f"l{layer}.o"))

    def forward(self, x: torch.Tensor, fb: ForwardBatch,
                kv_cache: Tuple[torch.Tensor, torch.Tensor],
                cos_sin: torch.Tensor) -> torch.Tensor:
        return self.o_proj(self.heads(x, fb, kv_cache, cos_sin))

    def heads(self, x: torch.Tensor, fb: ForwardBatch,
              kv_cache: Tuple[torch.Tensor, torch.Tensor],
              cos_sin: torch.Tensor) -> torch.Tensor:
        """What o_proj is applied to, [T, heads * head_dim]."""
        return self.attend(ops.linear(x, self.qkv, self.qkv_b), fb, kv_cache,
                           cos_sin)

    def attend(self, qkv: torch.Tensor, fb: ForwardBatch,
               kv_cache: Tuple[torch.Tensor, torch.Tensor],
               cos_sin: torch.Tensor) -> torch.Tensor:
        T = qkv.shape[0]
        # strided views into the fused QKV output — the HIP kernels take a
        # row stride, so there are no .contiguous() copies on the hot path
        q, k, v = qkv.split(
            [self.nq * self.hd, self.nkv * self.hd, self.nkv * self.hd], dim=-1)
        kc, vc = kv_cache
        if not fb.is_prefill:
            o = ops.rope_paged_attn_decode(
                fb.positions, q, k, v, cos_sin, kc, vc, fb.slot_mapping,
                fb.block_table, fb.ctx_lens, self.scale)
            return o.view(T, self.nq * self.hd)
        ops.rope_append(fb.positions, q, k, v, self.hd, cos_sin, kc, vc,
                        fb.slot_mapping)
        k3 = k.view(T, self.nkv, self.hd)
        v3 = v.view(T, self.nkv, self.hd)
        P = fb.num_prefill_tokens if fb.is_mixed else T
        qv = q.view(T, self.nq, self.hd)
        # prompt rows and decoded rows of a mixed round side by side
        o = qv.new_empty((T, self.nq, self.hd))
        if fb.prefix_lens is not None:
            # prefix-cache hit in the batch: q rows are suffixes;
            # cached prefix + the just-appended suffix K/V are read
            # back from the paged cache (ops/csrc/flash_prefill.hip)
            ops.flash_prefill_paged(
                qv[:P], kc, vc, fb.block_table,
                fb.prefix_lens, fb.cu_seqlens, fb.seq_lens, self.scale,
                out=o[:P])
        else:
            ops.flash_prefill(
                qv[:P], k3[:P], v3[:P], fb.cu_seqlens,
                fb.seq_lens, self.scale, out=o[:P])
        if fb.is_mixed:
            # mixed round: rows [P, T) are one decode token per
            # running sequence (engine._build_forward_batch)
            ops.paged_attn_decode(
                qv[P:], kc, vc, fb.decode_block_table,
                fb.decode_ctx_lens, self.scale, out=o[P:])
        return o.view(T, self.nq * self.hd)


class LlamaMLP(nn.Module):
    def __init__(self, cfg: ModelConfig, layer: int, device, dtype):
        super().__init__()
        tp, rank = tp_world_size(), tp_rank()
        h, inter = cfg.hidden_size, cfg.intermediate_size
        # gate and up fused in one column-parallel GEMM; the HIP silu_mul
        # kernel expects [gate | up] halves per shard
        self.gate_proj = ColumnParallelLinear(
            h, inter, rank, tp, device, dtype, _seed(f"l{layer}.gate"))
        self.up_proj = ColumnParallelLinear(
            h, inter, rank, tp, device, dtype, _seed(f"l{layer}.up"))
        self.down_proj = RowParallelLinear(
            inter, h, rank, tp, device, dtype, _seed(f"l{layer}.down"))
        # fuse gate+up into a single weight for one GEMM
        w = torch.cat([self.gate_proj.weight.data, self.up_proj.weight.data], 0)
        self.gate_up = nn.Parameter(w.contiguous(), requires_grad=False)
        del self.gate_proj, self.up_proj

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return self.down_proj(ops.linear_silu_mul(x, self.gate_up))


class LlamaLayer(nn.Module):
    def __init__(self, cfg: ModelConfig, layer: int, device, dtype):
        super().__init__()
        self.input_norm_w = nn.Parameter(
            torch.ones(cfg.hidden_size, dtype=dtype, device=device),
            requires_grad=False)
        self.post_norm_w = nn.Parameter(
            torch.ones(cfg.hidden_size, dtype=dtype, device=device),
            requires_grad=False)
        self.attn = LlamaAttention(cfg, layer, device, dtype)
        self.mlp = LlamaMLP(cfg, layer, device, dtype)
        self.eps = cfg.norm_eps

    def forward(self, x, residual, fb, kv_cache, cos_sin):
        if residual is None:
            residual = x.clone()
            x = ops.rmsnorm(x, self.input_norm_w, self.eps)
        else:
            x, residual = ops.fused_add_rmsnorm(
                x, residual, self.input_norm_w, self.eps)
        x = self.attn(x, fb, kv_cache, cos_sin)
        x, residual = ops.fused_add_rmsnorm(x, residual, self.post_norm_w,
                                            self.eps)
        x = self.mlp(x)
        return x, residual

    def opens(self) -> bool:
        """Whether normed and few_rows, which call none of the modules that they
        stand for, do what calls of them would."""
        attn, mlp = self._modules.get("attn"), self._modules.get("mlp")
        return (calls_plainly(self, LlamaLayer)
                and calls_plainly(attn, LlamaAttention)
                and calls_plainly(mlp, LlamaMLP)
                and calls_plainly(attn._modules.get("o_proj"),
                                  RowParallelLinear)
                and calls_plainly(mlp._modules.get("down_proj"),
                                  RowParallelLinear))

    def normed(self, x, residual, fb, kv_cache, cos_sin, next_norm_w):
        """x: the residual normed for this layer; returns it normed for what
        follows, by next_norm_w, and the residual."""
        x, residual = self.attn.o_proj.add_rmsnorm(
            self.attn.heads(x, fb, kv_cache, cos_sin), residual,
            self.post_norm_w, self.eps)
        return self.mlp.down_proj.add_rmsnorm(
            ops.linear_silu_mul(x, self.mlp.gate_up), residual, next_norm_w,
            self.eps)

    def few_rows(self, delta, residual, fb, kv_cache, cos_sin):
        """The layer for a few rows, whose products norm for themselves.  delta:
        what the residual still lacks (None: nothing); returns both."""
        qkv, residual = ops.norm_linear(
            delta, residual, self.input_norm_w, self.eps, self.attn.qkv,
            self.attn.qkv_b)
        delta = self.attn.o_proj(self.attn.attend(qkv, fb, kv_cache, cos_sin))
        act, residual = ops.norm_linear(
            delta, residual, self.post_norm_w, self.eps, self.mlp.gate_up,
            silu=True)
        return self.mlp.down_proj(act), residual


class LlamaForCausalLM(nn.Module):
    def __init__(self, cfg: ModelConfig, device, dtype=torch.bfloat16):
        super().__init__()
        self.cfg = cfg
        self.device = device
        self.embed = nn.Parameter(
            _init_weight((cfg.vocab_size, cfg.hidden_size), device, dtype,
                         _seed("embed")),
            requires_grad=False)
        self.layers = nn.ModuleList(
            LlamaLayer(cfg, i, device, dtype) for i in range(cfg.num_layers))
        self.final_norm_w = nn.Parameter(
            torch.ones(cfg.hidden_size, dtype=dtype, device=device),
            requires_grad=False)
        if cfg.tie_embeddings:
            self.lm_head = None
        else:
            self.lm_head = ReplicatedLinear(
                cfg.hidden_size, cfg.vocab_size, device, dtype,
                _seed("lm_head"))
        self.cos_sin = ops.build_cos_sin_cache(
            cfg.head_dim, cfg.max_position, cfg.rope_base, device=device,
            rope_scaling=cfg.rope_scaling)

    def forward(self, fb: ForwardBatch,
                kv_caches: List[Tuple[torch.Tensor, torch.Tensor]]
                ) -> torch.Tensor:
        residual = F.embedding(fb.token_ids, self.embed)
        if not all(layer.opens() for layer in self.layers):
            x, residual = residual, None
            for i, layer in enumerate(self.layers):
                x, residual = layer(x, residual, fb, kv_caches[i],
                                    self.cos_sin)
            return ops.fused_add_rmsnorm(x, residual, self.final_norm_w,
                                         self.cfg.norm_eps)[0]
        if residual.shape[0] <= FEW_ROWS:
            delta = None
            for i, layer in enumerate(self.layers):
                delta, residual = layer.few_rows(
                    delta, residual, fb, kv_caches[i], self.cos_sin)
            return ops.fused_add_rmsnorm(delta, residual, self.final_norm_w,
                                         self.cfg.norm_eps)[0]
        norms = [l.input_norm_w for l in self.layers] + [self.final_norm_w]
        x = ops.rmsnorm(residual, norms[0], self.cfg.norm_eps)
        for i, layer in enumerate(self.layers):
            x, residual = layer.normed(x, residual, fb, kv_caches[i],
                                       self.cos_sin, norms[i + 1])
        return x

    def compute_logits(self, hidden_last: torch.Tensor) -> torch.Tensor:
        """hidden_last: [B, hidden] -> bf16 logits [B, vocab] (the
        sampler's bf16 radix kernel consumes them directly)."""
        if self.lm_head is None:
            return ops.linear(hidden_last, self.embed)
        return self.lm_head(hidden_last)
