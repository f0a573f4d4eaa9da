"""Op dispatch: gfx950 HIP kernels on GPU tensors, torch reference on CPU.

Policy (driver contract): on a GPU box the HIP extension is REQUIRED — a
CUDA-device tensor with `_hip_ops` missing raises immediately rather than
silently falling back to eager torch. CPU tensors (tests, tiny gloo runs)
use ops.ref.
"""
import math
from typing import List, Optional, Tuple

import torch

from . import ref

try:
    from .. import _hip_ops as _ext
except ImportError:  # extension not built
    _ext = None


def hip_ops():
    """The raw extension module (router prefix kernels etc.). Fail-loud."""
    if _ext is None:
        raise RuntimeError(
            "_hip_ops extension is not built; run "
            "`python setup.py build_ext --inplace` (gfx950 HIP kernels are "
            "mandatory on GPU hosts — no eager fallback)")
    return _ext


def _use_hip(t: torch.Tensor) -> bool:
    if not t.is_cuda:
        return False
    hip_ops()  # raises if missing on a GPU path
    return True


def linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x @ w' of w [out, in]: few rows stream the weights through the HIP
    kernel, the rest is a library product."""
    return _ext.linear(x, w) if _use_hip(x) else x @ w.t()


def linear_parts(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """The same for rmsnorm or rope_and_cache, which also take the 32-bit
    partial sums [parts, rows, out] of a product that split K."""
    return _ext.linear_parts(x, w) if _use_hip(x) else x @ w.t()


def lay_weights(w: torch.Tensor) -> torch.Tensor:
    """Weights drawn as [in, out] in 32-bit -> bf16 [out, in] on the GPU."""
    return hip_ops().lay_weights(w)


def gated_linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """silu(x gate') * (x up') of w = [gate; up], mostly in one kernel."""
    if _use_hip(x):
        y = _ext.gated_linear(x, w, _SILU)
        if y is not None:
            return y
    return silu_mul(linear(x, w))


_SILU = 1       # activation code of the kernels


def _index(t: torch.Tensor, of: torch.Tensor) -> bool:
    """Whether the kernels take t as an index into rows of `of`."""
    return t.device == of.device and t.dim() == 1 and \
        t.dtype == torch.int64 and t.is_contiguous()


def rmsnorm(x: torch.Tensor, w: torch.Tensor, eps: float,
            residual: Optional[torch.Tensor] = None,
            rows: Optional[torch.Tensor] = None) -> torch.Tensor:
    """rows: the norms of these rows alone; what happens to the residual is
    left open then. A row that x does not have raises IndexError on the CPU and
    comes out as NaN on the GPU."""
    if _use_hip(x):
        if rows is None or (_index(rows, x) and x.shape[-1] % 8 == 0):
            return _ext.rmsnorm(x, w, eps, residual, rows)
        return _ext.rmsnorm(x, w, eps, residual)[rows]
    y = ref.rmsnorm(x, w, eps, residual)
    return y if rows is None else y[rows]


def embed_rmsnorm(ids: torch.Tensor, table: torch.Tensor, w: torch.Tensor,
                  eps: float):
    """-> table[ids] and its norm. An id that the table does not have raises
    IndexError on the CPU; on the GPU both of its rows come out as NaN."""
    if _use_hip(table) and _index(ids, table) and table.is_contiguous() and \
            table.dtype == torch.bfloat16 and table.shape[1] % 8 == 0:
        return _ext.embed_rmsnorm(ids, table, w, eps)
    x = table[ids]
    return x, rmsnorm(x, w, eps)


def rope(q: torch.Tensor, k: torch.Tensor, cos_sin: torch.Tensor,
         positions: torch.Tensor) -> None:
    if _use_hip(q):
        _ext.rope(q, k, cos_sin, positions.to(torch.int32))
        return
    ref.rope(q, k, cos_sin, positions)


def rope_and_cache(qkv: torch.Tensor, n_q_heads: int, cos_sin: torch.Tensor,
                   positions: torch.Tensor, k_cache: torch.Tensor,
                   v_cache: torch.Tensor, slots: torch.Tensor,
                   q_norm: Optional[torch.Tensor] = None,
                   k_norm: Optional[torch.Tensor] = None,
                   eps: float = 1e-5) -> torch.Tensor:
    """Packed heads of a qkv product (or its partial sums): q and k normed
    per head (where weights are given) and rotated, k and v stored in the
    cache. -> q [T, n_q_heads, D]."""
    if _use_hip(qkv):
        q = _ext.rope_and_cache(qkv, n_q_heads, cos_sin,
                                positions.to(torch.int32), k_cache, v_cache,
                                slots.to(torch.int64), q_norm, k_norm, eps)
        if q is not None:
            return q
        if qkv.dim() == 3:
            qkv = qkv.sum(0).to(torch.bfloat16)
    T, D, kvh = qkv.shape[0], k_cache.shape[3], k_cache.shape[1]
    q, k, v = (t.reshape(T, -1, D).contiguous() for t in qkv.split(
        [n_q_heads * D, kvh * D, kvh * D], dim=-1))
    if q_norm is not None:
        q = rmsnorm(q.view(-1, D), q_norm, eps).view(T, -1, D)
        k = rmsnorm(k.view(-1, D), k_norm, eps).view(T, -1, D)
    rope(q, k, cos_sin, positions)
    reshape_and_cache(k, v, k_cache, v_cache, slots)
    return q


def silu_mul(gate_up: torch.Tensor) -> torch.Tensor:
    if _use_hip(gate_up):
        return _ext.silu_mul(gate_up)
    return ref.silu_mul(gate_up)


def reshape_and_cache(k_new: torch.Tensor, v_new: torch.Tensor,
                      k_cache: torch.Tensor, v_cache: torch.Tensor,
                      slots: torch.Tensor) -> None:
    if _use_hip(k_new):
        _ext.reshape_and_cache(k_new, v_new, k_cache, v_cache,
                               slots.to(torch.int64))
        return
    ref.reshape_and_cache(k_new, v_new, k_cache, v_cache, slots)


def _one_round(groups: int) -> bool:
    """Whether parts of the decode attention can make up 5/6 of 256 workgroups, one
    round of 8 waves. By that / by 768 of 4 waves, us, 8 key heads of 4000 tokens, 8-bit
    and bf16: 9 sequences (84 %) 21.8 / 22.8, 32.4 / 32.8; 14 (88 %) 28.7 / 31.0, 47.2 /
    48.3; 16 30.3 / 33.4, 50.0 / 52.8; 13 (81 %) 28.2 / 27.1, 45.5 / 42.6; 12 (75 %)
    27.8 / 26.6, 44.4 / 42.0; 11 (69 %) 27.5 / 25.6, 44.0 / 38.5; 17 (53 %) 41.3 / 33.9,
    64.2 / 50.8; 21 (66 %) 46.8 / 39.0, 78.8 / 65.7."""
    return 256 // max(1, groups) * groups * 6 >= 256 * 5


def _past_a_round(groups: int, max_len: int, elem: int) -> bool:
    """Whether the decode attention has up to a quarter more workgroups than compute
    units, an eighth in 8 bits: some compute units then have two to do, and the others
    wait. Three parts of 4 waves, which a compute unit takes three of, even that out
    from where the sequences outweigh the second launch. One part / three, us, bf16:
    264 of 1000 tokens 36.5 / 34.2, of 4000 125 / 106; 320 of 500 22.9 / 24.9, of 1000
    37.6 / 36.3, of 4000 131 / 114, of 8000 272 / 235; 384 of 1500 58.0 / 58.3. 8-bit:
    264 of 700 16.8 / 18.5; 288 of 1500 30.5 / 31.7, of 2000 40.2 / 37.1, of 8000 141 /
    115; 320 of 4000 66.4 / 67.6."""
    if elem > 1:
        return 256 < groups <= 320 and max_len > 1024
    return 256 < groups <= 288 and max_len > 2048


def decode_parts(groups: int, max_len: int,
                 mean_len: Optional[float] = None,
                 elem: int = 2) -> Tuple[int, int]:
    """-> (parts, tokens per part) of the decode attention of `groups`
    (sequence, key head) pairs of up to max_len tokens, and of mean_len on
    average (None: 0.8 of that, lengths a quarter either way), of `elem` bytes a
    value. A workgroup of 8 waves takes 256 tokens a step, and a compute unit has
    registers for one of them or three of 4 waves: parts make up for fewer groups, by one
    round of the former (_one_round), or by at least one of the latter, as long as each
    has a step of its own. That is 768 workgroups, rounded up: the few of a second round
    cost less than the units that one part less leaves with two (us, up / down: 104
    groups of 2500 27.5 / 30.6, of 4000 39.2 / 42.6; 168 of 7000 109 / 119; 8-bit 58 /
    64; at the worst 176 of 7000 127 / 123).

    Parts cost their sums and a second launch. In us: one part takes 3 and as long as a
    workgroup walks (12.5 per 1000 tokens, 6.8 in 8 bits) or the bytes take at 5.2 TB/s,
    several 9 and the bytes at 5.8 TB/s. Over 264 batches of 1 to 24 sequences of like
    lengths, 8 key heads, the choice costs 0.2 % on average and 9 % at most; over 140,
    lengths alike to far apart, 0.4 and 24 %. One part / several, us, by groups and mean:
    8 of 400 6.7 / 8.3, of 800 11.2 / 9.1; 96 of 400 9.9 / 11.2, of 1500 24.9 / 21.6; 128
    of 1500 25.9 / 23.3; 136 of 2500 41.9 / 37.6; 152 of 1500 27.1 / 27.2, of 4000 72 /
    55; 168 of 1500 28.2 / 29.1, of 4000 76 / 67; 8-bit 136 of 2500 24.3 / 24.4, of 4000
    35.9 / 32.9; 168 of 4000 37.8 / 38.2, of 7000 66 / 58. From 200 groups on it is one
    (192 of 4000 80 / 80), but for _past_a_round.

    One long sequence among short ones would hold the batch up: 14 us per 1000
    tokens that a workgroup walks alone. It is cut so that none walks more than
    one and a half shares of a compute unit; up to 1000 tokens past these, or
    for less than twice the parts, the second launch costs as much. A sequence
    of 8000 among 24 of 100: 108 us in one part, 24 in 17; among 255 of 300: 258
    and 140 in 3; of 3000 among 16 of 300: 21 in 4, 17 in 8; of 1500 among 24 of
    1000: 27 in one, 34 in two."""
    parts = 1
    if groups < 200:
        walk = max_len * (12.5e-3 if elem > 1 else 6.8e-3)
        mean = 0.8 * max_len if mean_len is None else mean_len
        size = groups * mean * 256 * elem
        if 3 + max(walk, size / 5.2e6) > 9 + size / 5.8e6:
            parts = max(2, 256 // max(1, groups)) if _one_round(groups) \
                else -(-768 // max(1, groups))
    elif _past_a_round(groups, max_len, elem) and \
            (mean_len is None or max_len <= 1.4 * mean_len):
        parts = 3
    if mean_len is not None and max_len > 1.4 * mean_len:
        # tokens that one workgroup may walk while each compute unit takes one
        # and a half shares of the whole
        walk = max(256., 1.5 * mean_len * groups / 256)
        ragged = math.ceil(max_len / walk)
        if max_len - walk >= 1000 and ragged >= 2 * parts:
            parts = ragged
    parts = max(1, min(64, parts, -(-max_len // 256)))
    part = -(-(-(-max_len // parts)) // 32) * 32
    return -(-max_len // part), part


def decode_waves(groups: int, parts: int, max_len: int,
                 mean_len: Optional[float] = None, elem: int = 2,
                 apart: float = 2.) -> int:
    """Waves of a workgroup of the decode attention, 4 or 8; apart: how many times the
    mean the longest sequence may have where parts are shares of each sequence
    (else all have one length). Short sequences leave half of 8 without a tile (100
    sequences of 120 tokens: 19 us with 8 waves, 15 with 4). Where a compute unit has
    several workgroups to do, three of 4 waves have more under way than one of 8, which
    counts with few bytes a tile, and their ends overlap.

    In parts: as many as make that up (decode_parts), 0.88 of the time in geometric
    mean up to 1.4 times the mean (22 batches) and 0.92 up to 2 (23); past that 1.02.

    In one part: from 257 groups on, in 8 bits up to a mean of 1600 or up to 1024 tokens
    (8 / 4 waves, us: 40 of 600, 28 / 27, 8-bit 18.8 / 16.6; 100 of 300 32.4 / 28.2, 24.2
    / 18.6; 256 of 500 96 / 91, 71 / 53; 256 of 1500 252 / 257, 145 / 137; 32 of 300
    11.9 / 12.1, 10.1 / 10.2; 149 of 1640, 8-bit 98 / 104). But 4 waves walk the longest
    sequence twice as long as 8, and it is to end with the rest: with a compute unit's
    share of the tokens, and 400 (a launch and the first loads) beside it. 8-bit: 33
    sequences of 470 and one of 2494 20.5 / 29.5; 36 of 100 to 2100 25.0 / 29.6; 76 of
    up to 8190, 2800 on average 106 / 151; 106 of up to 3130, 770 on average 49 / 45. Over
    156 batches the choice costs 0.9 % on average and 14 % at most."""
    mean = 0.8 * max_len if mean_len is None else mean_len
    if max_len <= 256:
        return 4
    if parts > 1:
        many = groups < 200 and not _one_round(groups) or \
            _past_a_round(groups, max_len, elem)
        return 4 if many and (mean_len is None or max_len <= apart * mean) else 8
    few = mean <= 1600 if elem == 1 else max_len <= 1024
    return 4 if groups > 256 and few and \
        max_len <= 400 + 1.1 * groups * mean / 256 else 8


def decode_probe(max_len: int, mean_len: Optional[float], block: int) -> int:
    """The page that says whether sequences of the decode attention share their tokens:
    that at a third of the mean one. What they share is their first tokens; where that is
    more than a third, values are read by way of the caches (by way of them / past them,
    us, 256 sequences of 1500 tokens that share theirs by 8 prefixes, the first 500 217 /
    218, 8-bit 123 / 127; 750 195 / 206, 110 / 119; 1000 170 / 196, 97 / 112; none 271 /
    251, 150 / 138)."""
    mean = 0.8 * max_len if mean_len is None else mean_len
    return int(mean / 3) // block


def paged_attention(q: torch.Tensor, k_cache: torch.Tensor,
                    v_cache: torch.Tensor, block_tables: torch.Tensor,
                    seq_lens: torch.Tensor, scale: float,
                    max_seq_len: Optional[int] = None,
                    mean_seq_len: Optional[float] = None) -> torch.Tensor:
    if _use_hip(q):
        bt = block_tables.to(torch.int32)
        sl = seq_lens.to(torch.int32)
        waves, probe = 8, 0
        if max_seq_len is not None and max_seq_len > 0:
            probe = decode_probe(max_seq_len, mean_seq_len, k_cache.shape[2])
            groups, elem = q.shape[0] * k_cache.shape[1], k_cache.element_size()
            parts, part = decode_parts(groups, max_seq_len, mean_seq_len, elem)
            waves = decode_waves(groups, parts, max_seq_len, mean_seq_len, elem)
            if parts > 1:
                far_apart = mean_seq_len is not None and \
                    max_seq_len > 2 * mean_seq_len
                return _ext.paged_attention_split(q, k_cache, v_cache, bt,
                                                  sl, parts, part, scale,
                                                  waves=waves,
                                                  spread=far_apart,
                                                  probe=probe)
        return _ext.paged_attention(q, k_cache, v_cache, bt, sl, scale,
                                    waves=waves, probe=probe)
    return ref.paged_attention(q, k_cache, v_cache, block_tables, seq_lens,
                               scale)


def prefill_shape(news: List[int], ctxs: List[int], group: int,
                  kv_heads: int) -> int:
    """Shape of the prefill attention's workgroups (flash_prefill_bf16.hip) for
    prompts of `news` tokens that end contexts of `ctxs`: 0 by rows, 1 by keys,
    2 by rows with probabilities of 17 bits. From 256 workgroups by rows on the
    chip is full (1000 tokens behind 1000: 49 us by rows, 86 by keys). Below,
    the two with 17 bits are weighed in us, as measured: a workgroup by rows
    takes 5 + 0.026 per key, one by keys 5 + 0.0107, one per compute unit,
    those with the most keys first. One round of these is always faster."""
    rows = sum(-(-n * group // 128) for n in news) * kv_heads
    if rows >= 256:
        return 0
    some = [-(-n * group // 32) * kv_heads for n in news]
    if sum(some) <= 256:
        return 1
    work = sum(k * (5 + 0.0107 * (c - n / 2))
               for k, n, c in zip(some, news, ctxs)) / 256
    least = 5 + 0.0107 * min(c - n for n, c in zip(news, ctxs))
    most = max(ctxs)
    keys = 3 + max(5 + 0.0107 * most, work + 0.3 * least)
    return 1 if keys <= 5 + 0.026 * most else 2


def flash_prefill(q: torch.Tensor, k_cache: torch.Tensor,
                  v_cache: torch.Tensor, block_tables: torch.Tensor,
                  seq_meta: torch.Tensor, tiles: torch.Tensor,
                  scale: float, shape: int = -1) -> torch.Tensor:
    """Fused MFMA causal varlen prefill attention (GPU-only; callers fall
    back to the composed reference path when unsupported). shape: of its
    workgroups, from prefill_shape; below 0 by their number alone."""
    return hip_ops().flash_prefill(q, k_cache, v_cache, block_tables,
                                   seq_meta, tiles, scale, shape)


def move_blocks(pool: torch.Tensor, staging: torch.Tensor,
                block_ids: torch.Tensor, is_scatter: bool) -> None:
    if _use_hip(pool):
        _ext.move_blocks(pool, staging, block_ids.to(torch.int32), is_scatter)
        return
    # CPU reference: pool [L, 2, NB, KVH, BS, D]; staging [n, L, 2, KVH, BS, D]
    ids = block_ids.long()
    if is_scatter:
        pool[:, :, ids] = staging.permute(1, 2, 0, 3, 4, 5)
    else:
        staging.copy_(pool[:, :, ids].permute(2, 0, 1, 3, 4, 5))
