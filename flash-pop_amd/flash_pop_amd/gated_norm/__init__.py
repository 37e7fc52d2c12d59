"""gated_group_norm(retention, gate, eps=1e-6) -> bf16(GroupNorm_per_head(retention)) * bf16(swish(gate))

The step between the retention op and the output projection in the reference's layer
(flash_pop/retnet.py:294-309): GroupNorm with one group per head, computed in fp32, no affine
parameters (retnet.py:194-201), rounded to bf16, times swish(g_proj(x)) -- in one HIP launch
with the reference's rounding points.  retention [..., H, dv] (the op's output), gate [..., H*dv]
(the output of g_proj before the activation); returns [..., H*dv].  bfloat16 on the GPU;
dv = 8 * 2^k <= 512.  Gradients flow to both inputs (one launch).
"""
from .. import _lib, _ops


def gated_group_norm(retention, gate, eps: float = 1e-6):
    out = _lib.native().gated_group_norm(retention, gate, eps)
    if out is NotImplemented:
        if _ops.tracing():
            return _ops.Traced.apply(gated_group_norm, retention, gate, eps)
        _ops.check_gated_norm(retention, gate)
        _ops.rejected("gated_group_norm")
    return out
