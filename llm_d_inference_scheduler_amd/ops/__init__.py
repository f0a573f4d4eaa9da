from .dispatch import (  # noqa: F401
    flash_prefill, gated_linear, hip_ops, lay_weights, linear,
    move_blocks, paged_attention, reshape_and_cache, rmsnorm, rope, silu_mul,
)
