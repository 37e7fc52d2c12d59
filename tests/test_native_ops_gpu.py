"""The graph nodes of the native ops (csrc/torch_ops.cpp): which gradients arrive, outputs that nobody differentiates, saved
tensors that were changed in place, no_grad, several threads with a stream each."""
import threading

import pytest
import torch

import helpers as hp
import oracle

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("wanted", ["qkvs", "q", "s", "kv"])
@pytest.mark.parametrize("T", [70, 1100, 2001])   # 1100: the forward is cut into segments; 2001: the backward too
def test_gradients_of_some_inputs_from_some_outputs(wanted, T):
    from flash_pop_amd import fused_chunk_retention
    B, H, d = 1, 2, 64
    decays = oracle.head_decays(H)
    ins = dict(zip("qkvs", hp.make_inputs(B, T, H, d, d, seed=3, state_std=0.3, device=DEV)))
    d_o, d_s = hp.make_cotangents([(B, T, H, d), (B, H, d, d)], seed=4, device=DEV)
    for n in wanted:
        ins[n].requires_grad_()
    for use_o, use_s in ((True, True), (True, False), (False, True)):
        o, S = fused_chunk_retention(*ins.values(), decays)
        outs, cots = zip(*[(x, g) for x, g, use in ((o, d_o, use_o), (S, d_s, use_s)) if use])
        got = torch.autograd.grad(outs, [ins[n] for n in wanted], cots)
        _, _, ref = hp.oracle_plain(*[t.detach() for t in ins.values()], decays, d_o if use_o else torch.zeros_like(d_o), d_s if use_s else None)
        for n, g in zip(wanted, got):
            hp.assert_close(g, ref["qkvs".index(n)], f"d{n} from o={use_o} S={use_s}")


def test_no_grad_in_place_changes_and_reuse():
    from flash_pop_amd import XPos, flash_pop_retention, fused_chunk_retention, gated_group_norm
    q, k, v, s = hp.make_inputs(1, 70, 2, 64, 64, seed=5, state_std=0.3, device=DEV)
    decays = oracle.head_decays(2)
    q.requires_grad_()
    with torch.no_grad():
        assert not fused_chunk_retention(q, k, v, s, decays)[0].requires_grad
        assert not flash_pop_retention(q, k, v, s, decays, 32)[0].requires_grad
    o, _ = fused_chunk_retention(q, k, v, s, decays)
    v.add_(1)                                   # the node saved v
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        o.sum().backward()
    o, _ = fused_chunk_retention(q, k, v, s, decays)
    o.sum().backward()
    with pytest.raises(RuntimeError, match="second time"):
        o.sum().backward()
    # only one of the two rotated tensors is differentiated; a gate that needs no gradient
    k.requires_grad_()
    rq, rk = XPos(64)(q, k, 3)
    both = torch.autograd.grad([rq, rk], [q, k], [torch.ones_like(rq), torch.ones_like(rk)], retain_graph=True)
    assert torch.equal(torch.autograd.grad(rk, k, torch.ones_like(rk))[0], both[1])
    gate = torch.randn(1, 70, 128, device=DEV).to(hp.BF16)
    assert torch.autograd.grad(gated_group_norm(q, gate).sum(), q)[0].shape == q.shape


def test_saved_tensor_hooks_see_all_and_tangents_are_refused():
    from flash_pop_amd import XPos, flash_pop_retention, fused_chunk_retention, gated_group_norm
    decays = oracle.head_decays(2)
    q, k, v, s = hp.make_inputs(1, 2001, 2, 64, 64, seed=8, state_std=0.3, device=DEV)
    q.requires_grad_()
    for op, args in ((fused_chunk_retention, ()), (flash_pop_retention, (160,))):     # both cut into segments, both ways
        ref = torch.autograd.grad(op(q, k, v, s, decays, *args)[0].sum(), q)[0]
        packed = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.numel()) or t.cpu(), lambda t: t.to(DEV)):
            o, _ = op(q, k, v, s, decays, *args)
        assert len(packed) == 5                                                       # q, k, v, s and the segment states
        for _ in range(2):
            assert torch.equal(torch.autograd.grad(o.sum(), q, retain_graph=True)[0], ref)
    # (a block beyond the sequence is no block, however large)
    assert flash_pop_retention(q, k, v, s, decays, 2 ** 32)[1].shape[1] == 0
    import torch.autograd.forward_ad as fwd
    q = q.detach()
    with fwd.dual_level():
        dual = fwd.make_dual(q, torch.ones_like(q))
        for call in (lambda: fused_chunk_retention(dual, k, v, s, decays), lambda: flash_pop_retention(dual, k, v, s, decays, 64),
                     lambda: XPos(64)(dual, k, 0), lambda: gated_group_norm(dual, q.flatten(2))):
            with pytest.raises(NotImplementedError, match="forward mode"):
                call()


def test_threads_with_streams_of_their_own():
    from flash_pop_amd import fused_chunk_retention
    decays = oracle.head_decays(4)
    q, k, v, s = hp.make_inputs(2, 3001, 4, 64, 64, seed=6, state_std=0.3, device=DEV)   # cut into segments both ways
    d_o, = hp.make_cotangents([(2, 3001, 4, 64)], seed=7, device=DEV)

    def step():
        leaves = [t.detach().clone().requires_grad_() for t in (q, k, v, s)]
        o, _ = fused_chunk_retention(*leaves, decays)
        return o, *torch.autograd.grad(o, leaves, d_o)

    ref, bad = step(), []
    torch.cuda.synchronize()

    def work():
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(10):
                got = step()
                torch.cuda.current_stream().synchronize()
                bad.extend(i for i, (x, y) in enumerate(zip(got, ref)) if not torch.equal(x, y))

    threads = [threading.Thread(target=work) for _ in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
