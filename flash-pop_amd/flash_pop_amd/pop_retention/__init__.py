"""flash_pop_retention(q, k, v, s, head_decays, block_size) -> (o, block_states)

Same call signature and returns as the reference's FlashPOPRetention
(flash_pop/pop_retention/__init__.py:11-52): block_states is [B, T // block_size, H, dk, dv],
the recurrent state after every full block; there is no final-state output.  The block size
is kept on the autograd context, so T need not be a multiple of it in the backward pass
(the reference re-derives it as T // num_blocks, pop_retention/__init__.py:39-40).

flash_pop_retention_with_suffixes(q, k, v, s, head_decays, block_size, q_sfx, k_sfx, v_sfx)
    -> (o, o_sfx, last_state)

One POP layer step in a single walk: what POPDecoderLayer.pop_forward obtains from
flash_pop_retention followed by fused_chunk_retention on the suffix batch seeded with
[s, block_states] (flash_pop/pop_retnet.py:107-171), without writing the block states, reading
them back or concatenating them.  q_sfx, k_sfx, v_sfx are [B * (N + 1), Ls, H, d] with the block
index fastest (N = T // block_size, any Ls >= 1); last_state is the state after the last full
block, the reference's `states[:, -1]`.  Tokens after the last block boundary (T % block_size of
them) are context like any others; no suffix follows them.
"""
from .. import _lib, _ops


def _refused(q, k, v, s, head_decays, block_size):
    """Raises for arguments that the native ops did not take; -> the shape if it is the suffixes' fault."""
    block_size = int(block_size)
    assert block_size >= 1, f"block_size must be positive, got {block_size}"
    return _ops.check_retention(q, k, v, s, head_decays)


class FlashPOPRetention:
    """Stands for the reference's autograd Function of this name: `apply` is the op (forward, backward and graph node native)."""

    @staticmethod
    def apply(q, k, v, s, head_decays, block_size):
        out = _lib.native().flash_pop_retention(q, k, v, s, head_decays, block_size)
        if out is NotImplemented:
            if _ops.tracing():
                return _ops.Traced.apply(FlashPOPRetention.apply, q, k, v, s, head_decays, block_size)
            _refused(q, k, v, s, head_decays, block_size)
            _ops.rejected("flash_pop_retention")
        return out


flash_pop_retention = FlashPOPRetention.apply


class FlashPOPRetentionWithSuffixes:

    @staticmethod
    def apply(q, k, v, s, head_decays, block_size, q_sfx, k_sfx, v_sfx):
        out = _lib.native().flash_pop_retention_with_suffixes(q, k, v, s, head_decays, block_size, q_sfx, k_sfx, v_sfx)
        if out is NotImplemented:
            if _ops.tracing():
                return _ops.Traced.apply(FlashPOPRetentionWithSuffixes.apply, q, k, v, s, head_decays, block_size, q_sfx, k_sfx, v_sfx)
            shape = _refused(q, k, v, s, head_decays, block_size)
            _ops.check_suffixes(q_sfx, k_sfx, v_sfx, shape, int(block_size))
            _ops.rejected("flash_pop_retention_with_suffixes")
        return out


flash_pop_retention_with_suffixes = FlashPOPRetentionWithSuffixes.apply
