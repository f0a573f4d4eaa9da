from .dispatch import (  # noqa: F401
    embed_rmsnorm, flash_prefill, gated_linear, hip_ops, lay_weights, linear,
    linear_parts, move_blocks, paged_attention, prefill_shape,
    reshape_and_cache, rmsnorm, rope, rope_and_cache, silu_mul,
)
