"""The native ops (csrc/torch_ops.cpp) on the CPU: the same source, built over the CPU harness of the kernels, behind the
package's Python wrappers."""
import importlib.util
import os
import subprocess

import pytest
import torch

import helpers as hp
import oracle

EMU_DIR = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emu")
PKG_DIR = os.path.join(os.path.dirname(os.path.dirname(EMU_DIR)), "flash-pop_amd")
DEC = (0.97, 0.9)


def _module(name, path):
    spec = importlib.util.spec_from_file_location(name, path)
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


@pytest.fixture(scope="module")
def emu(tmp_path_factory):
    """(C-ABI library of the harness, the native ops over it)"""
    from flash_pop_amd import _lib
    lib = str(tmp_path_factory.mktemp("emu") / "libflashpop_emu.so")
    native = os.path.join(os.path.dirname(lib), "_native.so")
    build = _module("flash_pop_amd_build", os.path.join(PKG_DIR, "build.py"))
    ops = subprocess.Popen([os.path.join(EMU_DIR, "build_emu.sh")], env=dict(os.environ, EMU_OUT=lib))
    assert ops.wait() == 0
    subprocess.run(build.native_command(native, lib, EMU_DIR), check=True)
    return _lib.bind(lib), _module("_native", native)


@pytest.fixture
def ops(emu, monkeypatch):
    """The package, its wrappers over the harness"""
    import flash_pop_amd
    monkeypatch.setattr(flash_pop_amd._lib, "_native", emu[1])
    return flash_pop_amd


def _inputs(seed, B=1, T=70, H=2, d=64, block=32, Ls=3):
    q, k, v, s = hp.make_inputs(B, T, H, d, d, seed=seed, state_std=0.3)
    sfx = hp.make_suffix_inputs(B, T // block, Ls, H, d, d, seed=seed + 1)
    return q, k, v, s, sfx, torch.randn(B, T, H * d, generator=torch.Generator().manual_seed(seed)).to(hp.BF16)


def _calls(ops):
    """op -> (call of tensors alone, those tensors from a seed)"""
    xpos = ops.XPos(64)
    return {
        "plain": (lambda q, k, v, s: ops.fused_chunk_retention(q, k, v, s, DEC), lambda n: _inputs(n)[:4]),
        "pop": (lambda q, k, v, s: ops.flash_pop_retention(q, k, v, s, DEC, 32), lambda n: _inputs(n)[:4]),
        "pop_sfx": (lambda q, k, v, s, *x: ops.flash_pop_retention_with_suffixes(q, k, v, s, DEC, 32, *x), lambda n: (*_inputs(n)[:4], *_inputs(n)[4])),
        "rotary": (lambda q, k: xpos(q, k, 3), lambda n: _inputs(n)[:2]),
        "norm": (lambda q, g: ops.gated_group_norm(q, g), lambda n: (_inputs(n)[0], _inputs(n)[5])),
    }


OPS = ["plain", "pop", "pop_sfx", "rotary", "norm"]


def _tuple(out):
    return (out,) if isinstance(out, torch.Tensor) else out


@pytest.mark.parametrize("op", OPS)
@pytest.mark.filterwarnings("ignore")
def test_traced_programs_run_the_op_again(ops, op):
    """A program traced on some inputs gives, on others, what the op gives on those, gradients included."""
    call, inputs = _calls(ops)[op]
    traced = torch.jit.trace(call, tuple(inputs(1)))
    ins, ins2 = ([t.requires_grad_() for t in inputs(2)] for _ in range(2))
    out, ref = _tuple(traced(*ins)), _tuple(call(*ins2))
    assert all(torch.equal(a, b) for a, b in zip(out, ref))
    grads, ref = (torch.autograd.grad(x[0].sum(), y, allow_unused=True) for x, y in ((out, ins), (ref, ins2)))
    assert all((a is None and b is None) or torch.equal(a, b) for a, b in zip(grads, ref))
    with pytest.raises((RuntimeError, ValueError)):
        torch.jit.trace(call, (ins[0][:, :1], *ins[1:]))


@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.filterwarnings("ignore")
def test_traced_programs_run_the_decode_step_again(ops, in_place):
    step = lambda q, k, v, s: ops.retention_recurrent(q[:, 0], k[:, 0], v[:, 0], DEC, s, in_place=in_place)
    traced = torch.jit.trace(step, tuple(t.clone() for t in _inputs(1)[:4]), check_trace=False)
    ins, ins2 = _inputs(2)[:4], _inputs(2)[:4]
    out, ref = traced(*ins), step(*ins2)
    assert all(torch.equal(a, b) for a, b in zip((*out, ins[3]), (*ref, ins2[3])))
    assert (out[1].data_ptr() == ins[3].data_ptr()) == in_place


class _NoGradient(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x):
        return x.clone()

    @staticmethod
    def backward(ctx, g):
        return None


@pytest.mark.parametrize("op", OPS)
def test_gradients_are_zeros_where_nothing_arrives(ops, op):
    """Every input of an op gets a gradient: zeros where no output that depends on it is differentiated, or where what comes
    after the op passes nothing on."""
    call, inputs = _calls(ops)[op]
    ins = [t.requires_grad_() for t in inputs(1)]
    grads = torch.autograd.grad(_NoGradient.apply(_tuple(call(*ins))[0]).sum(), ins)
    assert all(g.shape == t.shape and not g.any() for g, t in zip(grads, ins))
    if op == "rotary":
        for i in (0, 1):
            grads = torch.autograd.grad(call(*ins)[i].sum(), ins)
            assert grads[i].any() and not grads[1 - i].any()
        call(*ins)[1].sum().backward()
        assert not ins[0].grad.any() and ins[1].grad.any()
        # an input that needs no gradient still gets none, and a lone q works
        assert torch.autograd.grad(call(ins[0], ins[1].detach())[0].sum(), ins[0])[0].any()
        assert torch.autograd.grad(ops.XPos(64)(ins[0], None, 0)[0].sum(), ins[0])[0].any()


def test_head_decays_are_what_has_a_length_and_floats(ops):
    q, k, v, s = _inputs(1)[:4]
    ref = ops.fused_chunk_retention(q, k, v, s, DEC)[0]
    for decays in (list(DEC), torch.tensor(DEC, dtype=torch.float64), [str(g) for g in DEC], dict.fromkeys(DEC)):
        assert torch.equal(ops.fused_chunk_retention(q, k, v, s, decays)[0], ref)
    for op in (lambda g: ops.fused_chunk_retention(q, k, v, s, g), lambda g: ops.retention_recurrent(q[:, 0], k[:, 0], v[:, 0], g, s)):
        for bad, error in (((g for g in DEC), TypeError), (DEC[0], TypeError), (("x", 0.5), ValueError), (DEC + DEC, AssertionError)):
            with pytest.raises(error):
                op(bad)


@pytest.mark.parametrize("op", OPS)
def test_second_derivatives_raise(ops, op):
    """create_graph gives the first derivative; what depends on it cannot be differentiated, and is not taken for a constant."""
    call, inputs = _calls(ops)[op]
    ins = [t.requires_grad_() for t in inputs(1)]
    first = lambda **kw: torch.autograd.grad(_tuple(call(*ins))[0].float().square().sum(), ins, allow_unused=True, **kw)
    grads = first(create_graph=True)
    assert all(torch.equal(a, b) for a, b in zip(grads, first()))
    penalty = ins[0].float().sum() + sum(g.float().square().sum() for g in grads)
    for differentiate in (lambda: penalty.backward(retain_graph=True), lambda: torch.autograd.grad(penalty, ins[0])):
        with pytest.raises(RuntimeError, match="once"):
            differentiate()


def test_positions_changed_before_the_backward_raise(ops):
    q, k = (t.requires_grad_() for t in _inputs(1, B=2)[:2])
    xpos, start = ops.XPos(64), torch.tensor([3, 5])
    out = xpos(q, k, start)[0].sum()
    ref = torch.autograd.grad(out, q, retain_graph=True)[0]
    start += 1
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(out, q)
    with torch.inference_mode():
        start = torch.tensor([3, 5])
    assert torch.equal(torch.autograd.grad(xpos(q, k, start)[0].sum(), q)[0], ref)
    # (positions of another type are converted, and the conversion is the op's own)
    start = torch.tensor([3, 5], dtype=torch.int32)
    out = xpos(q, k, start)[0].sum()
    start += 1
    assert torch.equal(torch.autograd.grad(out, q)[0], ref)


def test_in_place_steps_are_seen_by_the_graph(ops):
    q, k, v, s = _inputs(1)[:4]
    q.requires_grad_()
    out = ops.fused_chunk_retention(q, k, v, s, DEC)[0].sum()   # its node saves s
    step = lambda state, **kw: ops.retention_recurrent(q[:, 0], k[:, 0], v[:, 0], DEC, state, **kw)
    _, new = step(s)
    torch.autograd.grad(out, q, retain_graph=True)
    assert step(s, in_place=True)[1].data_ptr() == s.data_ptr() and torch.equal(s, new)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(out, q)
    with torch.inference_mode():
        state = s.clone()
    step(state, in_place=True)                                  # (has no version to advance)


@pytest.fixture
def launches_cost(emu):
    """launches_cost(steps): what the harness's device takes a launch for, so that not everything that can be cut is"""
    yield emu[0].emu_set_launch_steps
    emu[0].emu_set_launch_steps(0)


@pytest.mark.parametrize("T,block", [(650, 0), (326, 65)])
def test_only_what_the_backward_uses_is_kept(emu, ops, launches_cost, T, block):
    """The segment states of a cut forward go through the graph (and saved-tensor hooks) only if the backward is cut too; gradients
    are the oracle's either way."""
    lib, shape = emu[0], (1, T, 1, 64, 64) + ((block,) if block else ())
    name = "fp_pop_retention" if block else "fp_retention"
    forward, backward = getattr(lib, name + "_workspace_bytes"), getattr(lib, name + "_backward_workspace_bytes")
    q, k, v, s = hp.make_inputs(1, T, 1, 64, 64, seed=T, state_std=0.3)
    d_o, = hp.make_cotangents([(1, T, 1, 64)], seed=T)
    q.requires_grad_()
    call = (lambda: ops.flash_pop_retention(q, k, v, s, (0.97,), block)) if block else (lambda: ops.fused_chunk_retention(q, k, v, s, (0.97,)))
    ref = (hp.oracle_pop(q, k, v, s, (0.97,), block, d_o, None) if block else hp.oracle_plain(q, k, v, s, (0.97,), d_o, None))[2][0]
    seen = set()
    for steps in range(40):
        launches_cost(steps)
        cut = (forward(*shape) > 0, backward(*shape) > 0)
        if cut in seen or not cut[0]:
            continue
        seen.add(cut)
        packed = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t) or t, lambda t: t):
            out = call()[0]
        assert len(packed) == (5 if cut[1] else 4)
        hp.assert_close(torch.autograd.grad(out, q, d_o)[0], ref, f"dq, forward and backward cut: {cut}")
    # (the cut of a POP call always pays for its backward too at a size that the harness can run)
    assert seen == ({(True, True)} if block else {(True, True), (True, False)}), seen


def test_pass_ops_refuse_graph_capture(emu, ops):
    """Instantiating a HIP graph that holds the pass kernels has crashed the host process, so the retention ops raise, forward and
    backward, while their stream records one (the harness's flag: nothing is recorded).  The small kernels can be recorded."""
    calls = _calls(ops)
    ins = {op: [t.requires_grad_() for t in inputs(1)] for op, (_, inputs) in calls.items()}
    outs = {op: _tuple(call(*ins[op]))[0].sum() for op, (call, _) in calls.items()}
    x = [t.detach()[:, 0] for t in ins["plain"][:3]]
    emu[0].emu_set_capturing(1)
    try:
        for op, (call, _) in calls.items():
            for run in (lambda: call(*ins[op]), lambda: torch.autograd.grad(outs[op], ins[op], allow_unused=True)):
                if op in ("rotary", "norm"):
                    run()
                    continue
                with pytest.raises(RuntimeError, match="cannot be captured into a HIP graph"):
                    run()
        ops.retention_recurrent(*x, DEC, None)
    finally:
        emu[0].emu_set_capturing(0)
