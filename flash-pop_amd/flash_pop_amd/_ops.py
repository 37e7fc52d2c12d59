"""What the package's wrappers do around the native ops (csrc/torch_ops.cpp): those make their own checks of their arguments and leave
it to this module to say what was wrong; and the form of a call that torch.jit.trace can record."""
from __future__ import annotations

import torch


def check_devices(**tensors):
    for name, t in tensors.items():
        if t is not None and not t.is_cuda:
            raise RuntimeError(f"{name} is on {t.device}: flash_pop_amd runs on the GPU only")


def check_tensors(**tensors):
    for name, t in tensors.items():
        if t is not None:
            assert t.dtype == torch.bfloat16, f"{name}: only bfloat16 is supported, got {t.dtype}"
            check_devices(**{name: t})


def check_retention(q, k, v, s, head_decays):
    """Validate like the reference's asserts (fused_retention/__init__.py:20,
    pop_retention/__init__.py:17-18); -> (B, T, H, dk, dv)."""
    if q.dim() != 4 or k.shape != q.shape or v.dim() != 4 or v.shape[:3] != q.shape[:3]:
        raise ValueError(f"expected q, k [B,T,H,dk] and v [B,T,H,dv]; got {tuple(q.shape)}, {tuple(k.shape)}, {tuple(v.shape)}")
    B, T, H, dk = q.shape
    dv = v.shape[3]
    assert len(head_decays) == H, f"got {len(head_decays)} head decays for {H} heads"
    check_tensors(q=q, k=k, v=v, s=s)
    if s is not None and tuple(s.shape) != (B, H, dk, dv):
        raise ValueError(f"expected state [B,H,dk,dv] = {(B, H, dk, dv)}, got {tuple(s.shape)}")
    return B, T, H, dk, dv


def check_suffixes(q_sfx, k_sfx, v_sfx, shape, block_size):
    """Checks of the suffix batch as POPDecoderLayer._suffixes_forward makes them
    (flash_pop/pop_retnet.py:154-159): one suffix per block boundary, N + 1 per sequence."""
    B, T, H, dk, dv = shape
    n = B * (T // block_size + 1)
    if q_sfx.dim() != 4 or k_sfx.shape != q_sfx.shape or v_sfx.dim() != 4 or v_sfx.shape[:3] != q_sfx.shape[:3]:
        raise ValueError("expected q_sfx, k_sfx [B*(N+1),Ls,H,dk] and v_sfx [B*(N+1),Ls,H,dv]")
    if q_sfx.shape[0] != n or q_sfx.shape[2] != H or q_sfx.shape[3] != dk or v_sfx.shape[3] != dv:
        raise ValueError(f"got suffix tensors {tuple(q_sfx.shape)}, {tuple(v_sfx.shape)} for {n} suffixes of "
                         f"{H} heads with dk={dk}, dv={dv}: make sure there is one additional suffix block")
    check_tensors(q_sfx=q_sfx, k_sfx=k_sfx, v_sfx=v_sfx)


def check_decode_step(q, k, v, s, decays, in_place):
    """q, k [B,H,dk], v [B,H,dv], s [B,H,dk,dv] or None"""
    if q.dim() != 3 or k.shape != q.shape or v.dim() != 3 or v.shape[:2] != q.shape[:2]:
        raise ValueError(f"expected q, k [B,H,dk] and v [B,H,dv]; got {tuple(q.shape)}, {tuple(k.shape)}, {tuple(v.shape)}")
    B, H, dk = q.shape
    dv = v.shape[2]
    assert len(decays) == H, f"got {len(decays)} head decays for {H} heads"
    check_tensors(q=q, k=k, v=v, s=s)
    if s is not None and tuple(s.shape) != (B, H, dk, dv):
        raise ValueError(f"expected state [B,H,dk,dv] = {(B, H, dk, dv)}, got {tuple(s.shape)}")
    if in_place and (s is None or not s.is_contiguous()):
        raise ValueError("an in-place step needs a contiguous state tensor")


def check_rotary(q, k, theta, start):
    """q, k [B,T,H,d] (k may be None), theta [d / 2], start a number or a tensor [B]"""
    check_devices(q=q, k=k)
    check_tensors(q=q, k=k)
    if q.dim() != 4 or (k is not None and k.shape != q.shape):
        raise ValueError(f"expected q, k [B,T,H,d]; got {tuple(q.shape)}, {None if k is None else tuple(k.shape)}")
    B, d = q.shape[0], q.shape[3]
    if tuple(theta.shape) != (d // 2,) or theta.dtype != torch.float32 or theta.device != q.device:
        raise ValueError(f"theta must be {d // 2} floats on {q.device}")
    if isinstance(start, torch.Tensor) and (start.dim() != 1 or start.shape[0] != B):
        raise ValueError(f"start positions: expected one per sequence ({B}), got shape {tuple(start.shape)}")


def check_gated_norm(r, g):
    """r [..., H, dv], g [..., H * dv]"""
    check_devices(r=r, g=g)
    check_tensors(r=r, g=g)
    if r.dim() < 2 or g.numel() != r.numel() or g.shape[-1] != r.shape[-2] * r.shape[-1]:
        raise ValueError(f"expected r [..., H, dv] and g [..., H * dv]; got {tuple(r.shape)}, {tuple(g.shape)}")


def rejected(op):
    """The native op refused its arguments and the checks above found nothing to say about them."""
    raise TypeError(f"{op}: unsupported arguments")


class Traced(torch.autograd.Function):
    """An op as torch.jit.trace can record it: the tracer keeps calls of autograd Functions and runs them again, and does not see
    native ones.  apply(op, *op's arguments)."""

    @staticmethod
    def forward(ctx, op, *args):
        tracing = torch._C._get_tracing_state()
        torch._C._set_tracing_state(None)
        try:
            with torch.enable_grad():
                ctx.ins = [a.detach().requires_grad_(a.requires_grad) if isinstance(a, torch.Tensor) else a for a in args]
                out = op(*ctx.ins)
        finally:
            torch._C._set_tracing_state(tracing)
        ctx.set_materialize_grads(False)
        ctx.outs = (out,) if isinstance(out, torch.Tensor) else out
        detached = tuple(None if o is None else o.detach() for o in ctx.outs)
        return detached[0] if isinstance(out, torch.Tensor) else detached

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, *grads):
        if all(g is None for g in grads):
            return (None, *[torch.zeros_like(a) if isinstance(a, torch.Tensor) and a.requires_grad else None for a in ctx.ins])
        used = [(o, g) for o, g in zip(ctx.outs, grads) if g is not None]
        leaves = [a for a in ctx.ins if isinstance(a, torch.Tensor) and a.requires_grad]
        got = iter(torch.autograd.grad([o for o, _ in used], leaves, [g for _, g in used], retain_graph=True, allow_unused=True))
        return (None, *[next(got) if isinstance(a, torch.Tensor) and a.requires_grad else None for a in ctx.ins])


def tracing():
    return torch._C._get_tracing_state() is not None
