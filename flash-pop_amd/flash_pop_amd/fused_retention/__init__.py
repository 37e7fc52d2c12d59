"""fused_chunk_retention(q, k, v, s, head_decays) -> (o, s_out)

Same call signature and returns as the reference's FusedChunkRetention
(flash_pop/fused_retention/__init__.py:10-67): q, k [B,T,H,dk], v [B,T,H,dv], s [B,H,dk,dv],
all bfloat16 on the GPU; head_decays a tuple of H Python floats.  K is divided by sqrt(dk)
inside.  Gradients flow to q, k, v and s.  `s` may also be None (zeros), a superset of the
reference, whose callers substitute zeros themselves (flash_pop/retnet.py:279-282).
"""
from .. import _lib, _ops


class FusedChunkRetention:
    """Stands for the reference's autograd Function of this name: `apply` is the op.  Forward, backward and the graph node
    between them are native; the node saves what the reference saves (fused_retention/__init__.py:30) plus, where it pays, the
    states the forward passes through every few chunks."""

    @staticmethod
    def apply(q, k, v, s, head_decays):
        out = _lib.native().fused_chunk_retention(q, k, v, s, head_decays)
        if out is NotImplemented:
            if _ops.tracing():
                return _ops.Traced.apply(FusedChunkRetention.apply, q, k, v, s, head_decays)
            _ops.check_retention(q, k, v, s, head_decays)
            _ops.rejected("fused_chunk_retention")
        return out


fused_chunk_retention = FusedChunkRetention.apply
