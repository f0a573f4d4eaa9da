"""Llama-family model runner (random-init weights, paged KV, bf16).

MI355X-native execution path: projections of few rows stream their weights
through a HIP kernel, the rest go through hipBLASLt; the fused hot ops
(residual+RMSNorm, RoPE with the KV scatter, SiLU*up, GQA paged decode and
prefill attention) are the gfx950 HIP kernels in csrc/hip dispatched through
ops/. On the CPU, and for head sizes that the prefill kernels do not take,
prefill attention is composed of torch products over KV gathered from the paged
pool.

The reference router never runs a model — its pods do (vLLM). This runner
is the per-GPU worker engine's model, SURVEY.md §2.12 "worker shim".
"""
import math
from dataclasses import dataclass
from typing import Dict, List, Optional

import torch

from .. import ops
from ..ops import ref as ops_ref
from .configs import ModelConfig


@dataclass
class ForwardBatch:
    """One model invocation over a token-flattened batch.

    For decode: T == number of sequences, each contributing its newest token.
    For prefill: T == sum of chunk lengths; `seq_starts` delimits sequences.
    """
    input_ids: torch.Tensor          # [T] int64
    positions: torch.Tensor         # [T] int32
    slot_mapping: torch.Tensor      # [T] int64 into the paged pool
    is_decode: bool
    # decode-only:
    block_tables: Optional[torch.Tensor] = None   # [B, max_blocks] int32
    seq_lens: Optional[torch.Tensor] = None       # [B] int32 (incl. new token)
    max_seq_len: Optional[int] = None             # host-known max (no sync)
    mean_seq_len: Optional[float] = None          # and mean, if known
    # prefill-only:
    seq_starts: Optional[List[int]] = None        # len B+1 offsets into T
    ctx_lens: Optional[List[int]] = None          # [B] total ctx after chunk
    prefill_block_tables: Optional[List[torch.Tensor]] = None
    # fused flash-prefill metadata (GPU path; see flash_prefill.hip)
    prefill_bt: Optional[torch.Tensor] = None     # [S, max_blocks] int32
    prefill_meta: Optional[torch.Tensor] = None   # [S, 3] start,chunk,prior
    prefill_tiles: Optional[torch.Tensor] = None  # [n_tiles, 2] seq,vrow0
    logit_rows: Optional[torch.Tensor] = None     # rows needing logits
    # multimodal: rows whose input embedding is provided (encode hand-off)
    embed_rows: Optional[torch.Tensor] = None     # [n] int64 into T
    embed_values: Optional[torch.Tensor] = None   # [n, hidden]


class LlamaRunner:
    mixed_batches = False       # prefill and decode are passes of their own

    def __init__(self, config: ModelConfig, device: torch.device,
                 dtype: torch.dtype = torch.bfloat16, seed: int = 0):
        self.cfg = config
        self.device = device
        self.dtype = dtype
        self.scale = 1.0 / math.sqrt(config.head_dim)
        c = config
        if self.device.type == "cuda":
            # init directly on the GPU (16 GB of weights for Llama-3-8B —
            # CPU-side init would dominate startup). Same seed => identical
            # weights on every rank (required by the P/D KV hand-off).
            torch.cuda.manual_seed_all(seed)

            def draw(shape, std):
                return torch.empty(*shape, dtype=torch.float32,
                                   device=self.device).normal_(0.0, std)
        else:
            gen = torch.Generator(device="cpu").manual_seed(seed)

            def draw(shape, std):
                return torch.empty(*shape, dtype=torch.float32).normal_(
                    0.0, std, generator=gen)

        def w(*shape, std=0.02):
            return draw(shape, std).to(dtype).to(device)

        def linear(n_in, n_out, std=0.02):
            """[in, out] weights; on the GPU an output's weights lie together
            in memory: the streaming kernel needs that, and the library's
            large products run at 1490 TFLOP/s with it, 1280 without."""
            if self.device.type != "cuda" or dtype != torch.bfloat16:
                return w(n_in, n_out, std=std)
            return ops.lay_weights(draw((n_in, n_out), std)).t()

        out_std = 0.02 / math.sqrt(2 * c.num_layers)
        self.embed = w(c.vocab_size, c.hidden_size)
        self.layers: List[Dict[str, torch.Tensor]] = []
        for _ in range(c.num_layers):
            self.layers.append({
                "input_norm": torch.ones(c.hidden_size, dtype=dtype,
                                         device=device),
                "wqkv": linear(c.hidden_size, c.q_size + 2 * c.kv_size),
                "wo": linear(c.q_size, c.hidden_size, std=out_std),
                "post_norm": torch.ones(c.hidden_size, dtype=dtype,
                                        device=device),
                **({"q_norm": torch.ones(c.head_dim, dtype=dtype,
                                         device=device),
                    "k_norm": torch.ones(c.head_dim, dtype=dtype,
                                         device=device)}
                   if c.qk_norm else {}),
                "wgate_up": linear(c.hidden_size, 2 * c.intermediate_size),
                "wdown": linear(c.intermediate_size, c.hidden_size,
                                std=out_std),
            })
        self.final_norm = torch.ones(c.hidden_size, dtype=dtype, device=device)
        self.lm_head = self.embed if c.tie_embeddings else \
            w(c.vocab_size, c.hidden_size)
        self.cos_sin = ops_ref.rope_table(c.max_position, c.head_dim,
                                          c.rope_theta, device=device)

    def weight_bytes(self) -> int:
        total = self.embed.numel() + self.lm_head.numel() + \
            self.final_norm.numel()
        for layer in self.layers:
            total += sum(t.numel() for t in layer.values())
        return total * self.embed.element_size()

    # ------------------------------------------------------------------
    def forward(self, batch: ForwardBatch, kv_pool: torch.Tensor,
                embeddings_out: bool = False) -> torch.Tensor:
        """Returns logits [n_logit_rows, vocab] (or final hidden states for
        embeddings_out). kv_pool: [L, 2, NB, KVH, BS, D]."""
        c = self.cfg
        normed = residual = None
        if batch.embed_rows is not None and batch.embed_rows.numel():
            hidden = self.embed[batch.input_ids]
            hidden[batch.embed_rows] = batch.embed_values.to(hidden.dtype)
        elif self.layers:
            hidden, normed = ops.embed_rmsnorm(
                batch.input_ids, self.embed, self.layers[0]["input_norm"],
                c.rms_eps)
        else:
            hidden = self.embed[batch.input_ids]
        pos32 = batch.positions.to(torch.int32)
        shape = -1
        if batch.prefill_tiles is not None and batch.seq_starts and \
                batch.ctx_lens:
            shape = ops.prefill_shape(
                [e - s for s, e in zip(batch.seq_starts,
                                       batch.seq_starts[1:])],
                batch.ctx_lens, c.num_heads // c.num_kv_heads, c.num_kv_heads)
        for li, layer in enumerate(self.layers):
            if residual is None:
                residual = hidden
                if normed is None:
                    normed = ops.rmsnorm(hidden, layer["input_norm"],
                                         c.rms_eps)
            else:
                normed = ops.rmsnorm(hidden, layer["input_norm"], c.rms_eps,
                                     residual=residual)
            T = normed.shape[0]
            k_cache = kv_pool[li, 0]
            v_cache = kv_pool[li, 1]
            # Qwen3 norms every head of q and k before RoPE
            q = ops.rope_and_cache(
                ops.linear_parts(normed, layer["wqkv"].t()), c.num_heads,
                self.cos_sin, pos32, k_cache, v_cache, batch.slot_mapping,
                layer.get("q_norm"), layer.get("k_norm"), c.rms_eps)
            if batch.is_decode:
                attn = ops.paged_attention(q, k_cache, v_cache,
                                           batch.block_tables, batch.seq_lens,
                                           self.scale,
                                           max_seq_len=batch.max_seq_len,
                                           mean_seq_len=batch.mean_seq_len)
            else:
                attn = self._prefill_attention(batch, q, k_cache, v_cache,
                                               shape)
            o = ops.linear_parts(attn.view(T, c.q_size), layer["wo"].t())
            normed2 = ops.rmsnorm(o, layer["post_norm"], c.rms_eps,
                                  residual=residual)
            act = ops.gated_linear(normed2, layer["wgate_up"].t())
            hidden = ops.linear_parts(act, layer["wdown"].t())
        final = ops.rmsnorm(hidden, self.final_norm, c.rms_eps,
                            residual=residual,
                            rows=None if embeddings_out else batch.logit_rows)
        return final if embeddings_out else ops.linear(final, self.lm_head)

    def _prefill_attention(self, batch: ForwardBatch, q: torch.Tensor,
                           k_cache: torch.Tensor, v_cache: torch.Tensor,
                           shape: int = -1) -> torch.Tensor:
        """Causal varlen attention per sequence. GPU: fused MFMA flash
        kernel (flash_prefill.hip) — S never materialized. CPU fallback:
        composed chunked torch attention over pool-gathered KV."""
        c = self.cfg
        if (q.is_cuda and batch.prefill_tiles is not None
                and c.head_dim == 128
                and c.num_heads // c.num_kv_heads in (1, 2, 4, 8)):
            return ops.flash_prefill(
                q, k_cache, v_cache, batch.prefill_bt, batch.prefill_meta,
                batch.prefill_tiles, self.scale, shape)
        qpg = c.num_heads // c.num_kv_heads
        out = torch.empty_like(q)
        starts = batch.seq_starts
        for i in range(len(starts) - 1):
            s, e = starts[i], starts[i + 1]
            chunk = e - s
            ctx = batch.ctx_lens[i]
            prior = ctx - chunk
            kk, vv = ops_ref.gather_prefix(k_cache, v_cache,
                                           batch.prefill_block_tables[i], ctx)
            # [KVH, ctx, D]
            kk = kk.permute(1, 0, 2)
            vv = vv.permute(1, 0, 2)
            qi = q[s:e].view(chunk, c.num_kv_heads, qpg,
                             c.head_dim).permute(1, 2, 0, 3)  # [KVH,qpg,chunk,D]
            scores = torch.einsum("hgtd,hsd->hgts", qi.float(), kk.float())
            scores *= self.scale
            # causal mask: query t (global pos prior+t) sees keys <= prior+t
            t_idx = torch.arange(chunk, device=q.device).view(1, 1, chunk, 1)
            s_idx = torch.arange(ctx, device=q.device).view(1, 1, 1, ctx)
            scores.masked_fill_(s_idx > t_idx + prior, float("-inf"))
            p = torch.softmax(scores, dim=-1)
            o = torch.einsum("hgts,hsd->hgtd", p, vv.float())
            out[s:e] = o.permute(2, 0, 1, 3).reshape(
                chunk, c.num_heads, c.head_dim).to(q.dtype)
        return out
