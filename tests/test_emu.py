"""Runs the real kernel body and the real C-ABI layer on the CPU (one OS thread per GPU lane,
tests/emu/) and compares with the oracle.  This checks indexing, chunk scheduling, the pass
mapping and ragged/unaligned handling without a GPU; it assumes the documented MFMA lane
layout, which only the GPU parity tests can confirm."""
import ctypes
import os
import subprocess

import pytest
import torch

import helpers as hp
import oracle

EMU_DIR = os.path.join(os.path.dirname(os.path.abspath(__file__)), "emu")


@pytest.fixture(scope="module")
def emu_lib():
    subprocess.run([os.path.join(EMU_DIR, "build_emu.sh")], check=True)
    from flash_pop_amd import _lib
    return _lib.bind(os.path.join(EMU_DIR, "libflashpop_emu.so"))


@pytest.fixture
def choose_backward(emu_lib):
    """choose_backward(1 | 2): force the pass-per-gradient backward / the fused kernel for this test."""
    def choose(choice, every=-1):
        assert emu_lib.fp_set_backward_choice(choice, every) == 0
    yield choose
    assert emu_lib.fp_set_backward_choice(0, 512) == 0


PASSES, FUSED, PACED = 1, 2, 3
FOLD, WIDE = 22, 23   # two of the kernels' numbers in dispatch_pass


def _check_all(pairs):
    for name, got, ref in pairs:
        if ref is not None:
            hp.assert_close(got, ref, name)


@pytest.mark.parametrize("B,T,H,dk,dv,state_std", [
    (1, 150, 2, 128, 128, 0.5),     # ragged tail, initial state
    (1, 100, 2, 64, 128, None),     # dk != dv, no initial state
    (2, 64, 1, 128, 64, 0.0),       # exactly one chunk, zero state
    (1, 70, 1, 256, 64, 0.3),       # widest contraction (two visits per chunk), state stored as it is
    (1, 100, 1, 64, 256, 0.3),      # widest contraction in the dq and dk passes, state read transposed
    (1, 5, 3, 64, 64, 0.5),         # shorter than a chunk
    (5, 16, 1, 128, 128, 0.5),      # several short sequences per workgroup (suffix-like), odd count
    (5, 100, 1, 64, 128, None),     # several multi-chunk sequences per workgroup (the harness has 8 units), no initial state
    (1, 150, 1, 192, 64, 0.3),      # 192-wide keys: three visits per chunk in the forward and dv passes
    (1, 100, 2, 64, 192, 0.3),      # 192-wide values: three visits per chunk in the dq and dk passes
    (1, 130, 1, 192, 192, None),    # both, no initial state
])
def test_plain_fwd_bwd(emu_lib, B, T, H, dk, dv, state_std):
    decays = oracle.head_decays(H)
    q, k, v, s = hp.make_inputs(B, T, H, dk, dv, seed=T, state_std=state_std)
    d_o, d_s = hp.make_cotangents([(B, T, H, dv), (B, H, dk, dv)], seed=T + 1)
    o, S = hp.raw_fwd(emu_lib, q, k, v, s, decays)
    dq, dk_, dv_, ds0 = hp.raw_bwd(emu_lib, q, k, v, s, decays, d_o, d_s)
    o_ref, S_ref, (gq, gk, gv, gs) = hp.oracle_plain(q, k, v, s, decays, d_o, d_s)
    _check_all([("o", o, o_ref), ("S", S, S_ref), ("dq", dq, gq), ("dk", dk_, gk), ("dv", dv_, gv), ("ds0", ds0, gs)])


@pytest.mark.parametrize("B,T,H,dk,dv,block", [
    (1, 150, 2, 128, 128, 64),      # block == chunk
    (1, 287, 1, 64, 128, 144),      # block > chunk, ragged last block (reference generation shape)
    (2, 28, 1, 64, 64, 15),         # block < chunk
    (1, 130, 1, 64, 64, 32),        # block divides chunk
    (1, 40, 1, 64, 64, 100),        # no full block at all
    (1, 130, 1, 256, 64, 32),       # widest contraction with block states written and their gradients read
    (1, 130, 1, 192, 128, 48),      # three visits per chunk with block states
])
def test_pop_fwd_bwd(emu_lib, B, T, H, dk, dv, block):
    decays = oracle.head_decays(H, (5, 12))
    q, k, v, s = hp.make_inputs(B, T, H, dk, dv, seed=T + block, state_std=0.5)
    d_o, d_b = hp.make_cotangents([(B, T, H, dv), (B, T // block, H, dk, dv)], seed=T)
    o, states = hp.raw_pop_fwd(emu_lib, q, k, v, s, decays, block)
    dq, dk_, dv_, ds0 = hp.raw_pop_bwd(emu_lib, q, k, v, s, decays, block, d_o, d_b)
    o_ref, st_ref, (gq, gk, gv, gs) = hp.oracle_pop(q, k, v, s, decays, block, d_o, d_b)
    _check_all([("o", o, o_ref), ("states", states, st_ref), ("dq", dq, gq), ("dk", dk_, gk), ("dv", dv_, gv),
                ("ds0", ds0, gs)])


@pytest.mark.parametrize("B,T,H,dk,dv,block,state_std", [
    (1, 256, 1, 128, 128, 64, 0.5),     # a block state behind every chunk, the last one at the end of the sequence
    (1, 330, 2, 64, 128, 128, 0.5),     # two chunks per block, tokens after the last block boundary
    (1, 256, 1, 128, 64, 128, None),    # the sequence ends on a block boundary, no initial state
    (1, 300, 1, 64, 64, 192, 0.3),      # 64 x 64 states
    (1, 200, 1, 128, 128, 576, 0.5),    # no full block: nothing to add
])
def test_pop_backward_in_the_kernel_that_carries_ds_once(emu_lib, choose_backward, B, T, H, dk, dv, block, state_std):
    """flash_pop_retention's backward with whole chunks per block: the gradients of the block states join dS in the
    fused backward where its reverse walk crosses their boundaries.  Against the oracle and the pass-per-gradient path."""
    decays = oracle.head_decays(H, (5, 12))
    q, k, v, s = hp.make_inputs(B, T, H, dk, dv, seed=T + block, state_std=state_std)
    d_o, d_b = hp.make_cotangents([(B, T, H, dv), (B, T // block, H, dk, dv)], seed=T)
    choose_backward(FUSED)
    grads = hp.raw_pop_bwd(emu_lib, q, k, v, s, decays, block, d_o, d_b)
    _, _, ref = hp.oracle_pop(q, k, v, s, decays, block, d_o, d_b)
    _check_all([(n, g, r) for n, g, r in zip(("dq", "dk", "dv", "ds0"), grads, ref)])
    choose_backward(PASSES)
    other = hp.raw_pop_bwd(emu_lib, q, k, v, s, decays, block, d_o, d_b)
    assert not all(torch.equal(x, y) for x, y in zip(grads, other) if x is not None), "both calls took the same kernels"
    for n, x, y in zip(("dq", "dk", "dv", "ds0"), grads, other):
        if x is not None:
            assert hp.error_report(x, y.float())["rms_ratio"] < 0.004, n


FUSED_NAMES = ("dq", "dk", "dv", "dq_sfx", "dk_sfx", "dv_sfx", "ds0")


@pytest.mark.parametrize("B,nblk,block,Ls,H,dk,dv,state_std,tail", [
    (1, 2, 64, 16, 2, 128, 128, 0.5, 0),    # block == chunk
    (2, 2, 80, 5, 1, 64, 128, None, 0),     # block of a full and a short chunk, no initial state
    (1, 3, 24, 64, 1, 128, 64, 0.5, 0),     # block shorter than a chunk, suffix as long as one
    (1, 1, 130, 1, 1, 64, 64, 0.0, 0),      # one block of three chunks, one-token suffixes
    (1, 2, 40, 9, 1, 256, 64, 0.5, 0),      # two visits per chunk in the forward and dv passes
    (1, 2, 64, 16, 1, 64, 256, 0.5, 0),     # ... in the dq and dk passes
    (2, 2, 64, 16, 1, 128, 128, 0.5, 37),   # tokens after the last block boundary (less than a chunk)
    (1, 1, 150, 7, 2, 64, 128, None, 100),  # ... more than a chunk of them, no initial state
    (1, 0, 90, 12, 1, 64, 64, 0.5, 70),     # no full block at all: one suffix, read from the initial state
    (1, 2, 40, 9, 1, 256, 64, 0.5, 11),     # ... with two visits per chunk
    (1, 2, 64, 100, 1, 128, 128, 0.5, 0),   # suffixes longer than a chunk: two parts
    (1, 1, 80, 130, 2, 64, 128, None, 30),  # ... three parts, tokens after the last boundary, no initial state
    (1, 1, 64, 128, 1, 64, 128, 0.3, 0),    # ... two full parts, dk != dv
    (1, 2, 40, 9, 1, 192, 64, 0.5, 0),      # three visits per chunk in the forward and dv passes
    (1, 2, 40, 9, 1, 128, 192, 0.5, 13),    # ... in the dq and dk passes, with trailing tokens
])
def test_fused_pop_fwd_bwd(emu_lib, B, nblk, block, Ls, H, dk, dv, state_std, tail):
    decays = oracle.head_decays(H, (4, 9))
    T = nblk * block + tail
    q, k, v, s = hp.make_inputs(B, T, H, dk, dv, seed=T + Ls, state_std=state_std)
    sfx = hp.make_suffix_inputs(B, nblk, Ls, H, dk, dv, seed=T + Ls + 1)
    cot = hp.make_cotangents([(B, T, H, dv), tuple(sfx[2].shape), (B, H, dk, dv)], seed=T + 2)
    o, o_sfx, S = hp.raw_fused_fwd(emu_lib, q, k, v, s, sfx, decays, block)
    grads = hp.raw_fused_bwd(emu_lib, q, k, v, s, sfx, decays, block, cot)
    o_ref, os_ref, S_ref, g_ref = hp.oracle_fused(q, k, v, s, sfx, decays, block, cot)
    _check_all([("o", o, o_ref), ("o_sfx", o_sfx, os_ref), ("s_out", S, S_ref)])
    _check_all([(n, g, r) for n, g, r in zip(FUSED_NAMES, grads, g_ref)])


@pytest.mark.parametrize("B,nblk,block,Ls,H,dv,state_std", [
    (1, 3, 65, 16, 1, 64, 0.5),      # a chunk of one token per block
    (1, 2, 128, 1, 1, 192, None),    # two chunks per block, one-token suffixes, three column tiles, no initial state
    (2, 4, 15, 15, 2, 64, 0.5),      # blocks shorter than a row block
    (1, 1, 63, 16, 1, 128, 0.5),     # a single short block
    (1, 8, 65, 16, 1, 64, 0.5),      # more chunks than are under way: of one token per block
    (1, 8, 96, 1, 2, 64, None),      # ... of half a chunk, one-token suffixes, two heads, no initial state
    (1, 4, 63, 16, 1, 192, 0.5),     # ... blocks of less than a chunk, three column tiles
    (3, 3, 15, 15, 1, 256, 0.5),     # ... twelve workgroups on eight units
])
def test_folded_forward(emu_lib, B, nblk, block, Ls, H, dv, state_std):
    """64-wide keys and short suffixes: taken as part of the chunks at their boundaries."""
    assert emu_lib.emu_pop_folds(B, nblk * block, H, 64, dv, block, Ls, 8) == 1
    assert emu_lib.emu_pass_kernel(1, B, nblk * block, H, 64, dv, block, Ls, 0, 8) == FOLD
    decays = oracle.head_decays(H, (4, 9))
    q, k, v, s = hp.make_inputs(B, nblk * block, H, 64, dv, seed=block + Ls, state_std=state_std)
    sfx = hp.make_suffix_inputs(B, nblk, Ls, H, 64, dv, seed=block + Ls + 1)
    o, o_sfx, S = hp.raw_fused_fwd(emu_lib, q, k, v, s, sfx, decays, block)
    cot = hp.make_cotangents([tuple(v.shape), tuple(sfx[2].shape), (B, H, 64, dv)], seed=1)
    o_ref, os_ref, S_ref, _ = hp.oracle_fused(q, k, v, s, sfx, decays, block, cot)
    _check_all([("o", o, o_ref), ("o_sfx", o_sfx, os_ref), ("s_out", S, S_ref)])


@pytest.mark.parametrize("folds,B,nblk,H,dk,dv,block,Ls", [
    (1, 8, 32, 12, 64, 128, 64, 16),
    (1, 8, 1, 12, 64, 128, 64, 16),       # a single block
    (1, 8, 3, 12, 64, 128, 33, 16),
    (1, 8, 4, 12, 64, 128, 64, 16),
    (1, 8, 3, 12, 64, 256, 32, 16),
    (1, 8, 2, 12, 64, 256, 1, 1),
    (1, 8, 7, 8, 64, 128, 72, 3),         # two chunks a block
    (1, 8, 8, 8, 64, 128, 96, 3),
    (1, 8, 8, 8, 64, 256, 104, 3),
    (1, 8, 64, 8, 64, 256, 105, 3),
    (1, 4, 64, 8, 64, 64, 97, 3),
    (1, 4, 4, 32, 64, 64, 64, 16),        # 64 x 64 states
    (1, 129, 11, 1, 64, 64, 64, 16),      # ... where the bytes count
    (1, 129, 12, 1, 64, 64, 64, 16),
    (1, 17, 3, 8, 64, 64, 32, 16),
    (1, 17, 4, 8, 64, 64, 32, 16),
    (1, 17, 3, 8, 64, 64, 16, 16),
    (1, 17, 11, 8, 64, 64, 80, 16),
    (1, 17, 12, 8, 64, 64, 80, 16),
    (0, 8, 32, 12, 128, 128, 64, 16),     # never: 128-wide keys, longer suffixes
    (0, 8, 32, 12, 64, 128, 64, 17),
])
def test_rule_of_the_folded_forward(emu_lib, folds, B, nblk, H, dk, dv, block, Ls):
    """Which POP calls with suffixes go to the folding kernel, at 256 units: those that it is faster at."""
    assert emu_lib.emu_pop_folds(B, nblk * block, H, dk, dv, block, Ls, 256) == folds
    if block > 1:
        assert emu_lib.emu_pop_folds(B, nblk * block + 1, H, dk, dv, block, Ls, 256) == 0   # tokens after the last boundary


@pytest.mark.parametrize("kernel,T,dk,dv,block,Ls", [
    *[(FOLD, nblk * block, 64, dv, block, Ls) for dv in (64, 128, 256) for nblk, block, Ls in ((1, 1, 1), (1, 64, 16), (2, 105, 3), (64, 64, 16))],
    (0, 2048, 64, 128, 64, 17),      # longer suffixes
    (14, 2049, 64, 128, 64, 16),     # tokens after the last boundary
    (5, 2048, 128, 128, 64, 16),     # 128-wide keys
])
def test_kernel_of_a_forward_with_suffixes(emu_lib, kernel, T, dk, dv, block, Ls):
    """Which POP calls with suffixes have them folded: those whose suffixes fit, whatever the number of blocks, streams and units.  Never
    walking backward."""
    for B, H, units in ((1, 1, 256), (8, 12, 256), (129, 1, 256), (1, 1, 8)):
        assert emu_lib.emu_pass_kernel(1, B, T, H, dk, dv, block, Ls, 0, units) == kernel
    assert emu_lib.emu_pass_kernel(1, 8, T, 12, dk, dv, block, Ls, 1, 256) == (0 if kernel == FOLD else kernel)


@pytest.mark.parametrize("kernel,passes,B,T,H,dk,dv,block", [
    (9, 1, 128, 2048, 1, 128, 128, 0),      # 128 columns per workgroup on half of the units: 64 columns each fit at once
    (WIDE, 1, 129, 2048, 1, 128, 128, 0),
    (9, 1, 4, 2048, 16, 128, 256, 0),
    (WIDE, 1, 5, 1, 16, 128, 256, 0),       # any length while those of 128 columns fit
    (9, 2, 64, 2048, 1, 128, 128, 0),       # two passes share a launch
    (WIDE, 2, 65, 2048, 1, 128, 128, 0),
    (WIDE, 3, 43, 2048, 1, 128, 128, 0),
    (WIDE, 1, 256, 1, 1, 128, 128, 0),
    (8, 1, 257, 383, 1, 128, 128, 0),       # more: sequences that are worth a workgroup
    (WIDE, 1, 257, 384, 1, 128, 128, 0),
    (8, 1, 129, 191, 1, 128, 256, 0),
    (WIDE, 1, 129, 192, 1, 128, 256, 0),
    (8, 1, 257, 4096, 1, 128, 192, 0),      # no whole number of 128 columns
    (8, 1, 257, 4096, 1, 128, 64, 0),
    (6, 1, 257, 4096, 1, 128, 128, 64),     # block states
    (11, 1, 257, 4096, 1, 256, 128, 0),     # other keys
    (1, 1, 257, 4096, 1, 64, 128, 64),
    (3, 1, 129, 4096, 1, 64, 128, 0),
    (4, 1, 128, 4096, 1, 64, 128, 0),
])
def test_rule_of_128_columns_per_workgroup(emu_lib, kernel, passes, B, T, H, dk, dv, block):
    """Which passes run with 128 columns per workgroup, at 256 units, in either direction."""
    for reverse in (0, 1):
        assert emu_lib.emu_pass_kernel(passes, B, T, H, dk, dv, block, 0, reverse, 256) == kernel


@pytest.mark.parametrize("B,T,H,dk,dv,state_std,segments", [
    (1, 512, 1, 64, 64, 0.5, 2),       # the harness pretends to have 8 compute units: 1 stream -> 2 segments of 4 chunks
    (1, 1024, 1, 64, 128, None, 4),    # dk != dv, no initial state, 4 segments
    (1, 256, 1, 64, 64, 0.5, 1),       # too short to cut: same path as the plain entry point
    (1, 512, 1, 256, 64, 0.5, 2),      # 256-wide keys: the state-only walk visits every chunk twice
    (1, 512, 1, 192, 64, 0.5, 2),      # 192-wide keys: three visits
    (1, 640, 1, 128, 128, 0.5, 2),     # 128-wide keys: the state-only kernel with the whole state tile per workgroup, 5 chunks
    (1, 512, 1, 128, 256, None, 2),    # ... two workgroups per sequence (256-wide values), 4 chunks per segment
])
def test_split_sequences_fwd_bwd(emu_lib, B, T, H, dk, dv, state_std, segments):
    decays = (0.97,) * H
    q, k, v, s = hp.make_inputs(B, T, H, dk, dv, seed=T, state_std=state_std)
    d_o, d_s = hp.make_cotangents([(B, T, H, dv), (B, H, dk, dv)], seed=T + 1)
    o, S, nbytes = hp.raw_split_fwd(emu_lib, q, k, v, s, decays)
    assert nbytes == (2 * 2 * B * segments * H * dk * dv if segments > 1 else 0)
    dq, dk_, dv_, ds0 = hp.raw_split_bwd(emu_lib, q, k, v, s, decays, d_o, d_s)
    o_ref, S_ref, (gq, gk, gv, gs) = hp.oracle_plain(q, k, v, s, decays, d_o, d_s)
    _check_all([("o", o, o_ref), ("S", S, S_ref), ("dq", dq, gq), ("dk", dk_, gk), ("dv", dv_, gv), ("ds0", ds0, gs)])
    # the backward that starts from the segment states the forward left in its workspace: same bits
    o2, S2, _, ws = hp.raw_split_fwd(emu_lib, q, k, v, s, decays, keep_workspace=True)
    again = hp.raw_split_bwd(emu_lib, q, k, v, s, decays, d_o, d_s, forward_workspace=ws)
    assert torch.equal(o2, o) and all(torch.equal(a, b) for a, b in zip(again, (dq, dk_, dv_, ds0)))


@pytest.mark.parametrize("B,T,H,dk,dv,state_std,segments,gamma", [
    (1, 257, 1, 64, 64, 0.5, 2, 0.9),       # the last segment is one token
    (1, 511, 1, 128, 128, 0.5, 2, 0.9),     # one token short of two whole segments: a short last chunk in the state-only kernel
    (1, 700, 1, 64, 128, None, 3, 0.9),     # 11 chunks, the last one short, no initial state
    (1, 704, 1, 64, 64, 0.5, 3, 0.9),       # 11 whole chunks in segments of 4, 4 and 3
    (2, 300, 1, 128, 128, 0.5, 1, 0.9),     # too many streams for the harness's 8 units: not cut
    (1, 300, 1, 128, 256, 0.3, 2, 0.9),     # two workgroups per segment in the state-only kernel
    (1, 330, 1, 256, 64, 0.3, 2, 0.9),      # the state-only walk visits every chunk twice
    (2, 330, 1, 64, 64, 0.5, 2, 0.9),       # rows of the second sequence start inside a chunk
    (1, 700, 1, 64, 64, 0.5, 3, 0.99),
    (1, 620, 1, 128, 128, 0.5, 3, 0.99),
])
def test_split_sequences_uneven(emu_lib, B, T, H, dk, dv, state_std, segments, gamma):
    """Sequences that do not fall into equal segments of whole chunks, with a decay strong enough that a state one token off
    would show, and with one that leaves something of a state over a whole segment (0.99^256 = 0.08)."""
    decays = (gamma,) * H
    q, k, v, s = hp.make_inputs(B, T, H, dk, dv, seed=T, state_std=state_std)
    d_o, d_s = hp.make_cotangents([(B, T, H, dv), (B, H, dk, dv)], seed=T + 1)
    o, S, nbytes, ws = hp.raw_split_fwd(emu_lib, q, k, v, s, decays, keep_workspace=True)
    assert nbytes == (2 * 2 * B * segments * H * dk * dv if segments > 1 else 0)
    dq, dk_, dv_, ds0 = hp.raw_split_bwd(emu_lib, q, k, v, s, decays, d_o, d_s, forward_workspace=ws if segments > 1 else None)
    o_ref, S_ref, (gq, gk, gv, gs) = hp.oracle_plain(q, k, v, s, decays, d_o, d_s)
    _check_all([("o", o, o_ref), ("S", S, S_ref), ("dq", dq, gq), ("dk", dk_, gk), ("dv", dv_, gv), ("ds0", ds0, gs)])
    # the states between the segments carry 16 bits more than bf16: not further from the oracle than the uncut call
    o1, S1 = hp.raw_fwd(emu_lib, q, k, v, s, decays)
    grads1 = hp.raw_bwd(emu_lib, q, k, v, s, decays, d_o, d_s)
    for name, got, uncut, ref in zip(("o", "S", "dq", "dk", "dv", "ds0"), (o, S, dq, dk_, dv_, ds0), (o1, S1, *grads1),
                                     (o_ref, S_ref, gq, gk, gv, gs)):
        if ref is not None:
            assert oracle.rms_error_ratio(got.float(), ref) <= 1.05 * oracle.rms_error_ratio(uncut.float(), ref), name


@pytest.mark.parametrize("B,T,H,dk,dv,block,state_std,segments", [
    (1, 256, 1, 128, 128, 64, 0.5, 4),     # whole chunks per block, the sequence ends on a boundary
    (1, 287, 1, 64, 128, 144, 0.5, 2),     # blocks that end inside a chunk, tokens after the last one
    (2, 211, 1, 64, 64, 70, None, 4),      # one token after the last block, no initial state, two sequences
    (1, 200, 1, 128, 64, 100, 0.3, 2),
    (1, 150, 1, 256, 64, 65, 0.3, 3),      # the state-only walk visits every chunk twice
    (1, 200, 1, 64, 64, 32, 0.5, 1),       # blocks shorter than a chunk: not cut
    (1, 64, 1, 64, 64, 64, 0.5, 1),        # a single block
])
def test_pop_split_at_blocks(emu_lib, B, T, H, dk, dv, block, state_std, segments):
    decays = (0.97,) * H
    q, k, v, s = hp.make_inputs(B, T, H, dk, dv, seed=T + block, state_std=state_std)
    d_o, d_b = hp.make_cotangents([(B, T, H, dv), (B, T // block, H, dk, dv)], seed=T)
    nbytes = emu_lib.fp_pop_retention_workspace_bytes(B, T, H, dk, dv, block)
    assert nbytes == (2 * 2 * B * segments * H * dk * dv if segments > 1 else 0)
    ws = torch.empty(max(nbytes, 16), dtype=torch.uint8)
    p, dec = hp._p, hp._dec(decays)
    nan = lambda *shape: torch.full(shape, float("nan"), dtype=hp.BF16)
    o, states = nan(B, T, H, dv), nan(B, T // block, H, dk, dv)
    assert emu_lib.fp_pop_retention_fwd_split(p(q), p(k), p(v), p(s), dec, p(o), p(states), B, T, H, dk, dv, block, p(ws), nbytes, None) == 0
    o_ref, st_ref, refs = hp.oracle_pop(q, k, v, s, decays, block, d_o, d_b)
    o1, states1 = hp.raw_pop_fwd(emu_lib, q, k, v, s, decays, block)
    grads1 = hp.raw_pop_bwd(emu_lib, q, k, v, s, decays, block, d_o, d_b)
    for kept in (1, 0):   # from the states that the forward left, and from recomputed ones
        grads = [nan(*q.shape), nan(*k.shape), nan(*v.shape), nan(B, H, dk, dv)]
        assert emu_lib.fp_pop_retention_bwd_split(p(q), p(k), p(v), p(s), dec, p(d_o), p(d_b), *[p(g) for g in grads], B, T, H, dk, dv,
                                                  block, p(ws), nbytes, kept, None) == 0
        names, got, uncut = ("o", "states", "dq", "dk", "dv", "ds0"), (o, states, *grads), (o1, states1, *grads1)
        for name, g, u, ref in zip(names, got, uncut, (o_ref, st_ref, *refs)):
            if ref is None:
                continue
            hp.assert_close(g, ref, name)
            # both halves of the states between the blocks: not further from the oracle than the uncut call
            assert oracle.rms_error_ratio(g.float(), ref) <= 1.05 * oracle.rms_error_ratio(u.float(), ref), name
    if nbytes:   # argument checks come before any launch
        rc = lambda w, n: emu_lib.fp_pop_retention_fwd_split(p(q), p(k), p(v), p(s), dec, p(o), p(states), B, T, H, dk, dv, block, w, n, None)
        assert rc(None, 0) == -1 and b"fp_pop_retention_workspace_bytes" in emu_lib.fp_last_error()
        assert rc(p(ws), nbytes - 16) == -2 and b"fp_pop_retention_workspace_bytes" in emu_lib.fp_last_error()


@pytest.mark.parametrize("T,dk,dv,block", [
    (256, 128, 128, 64),   # POP cut at its blocks, 128-wide keys
    (150, 256, 64, 64),    # the same through the state-only kernel for 64-row states, a tail after the last block
    (330, 256, 64, 0),     # the plain op in uneven segments
])
def test_cut_calls_carry_fp32_states(emu_lib, choose_backward, T, dk, dv, block):
    """A cut call hands its states from launch to launch as fp32, so that it differs from the uncut one by the order of
    fp32 sums alone.  A state element that moved by a few 2^-24 rounds to another bf16 operand in about one case of 2^13;
    an output reads dk of them (1.5 % to 3 % have one that moved), and one operand off by half a bf16 step moves a sum of dk
    such terms across a rounding boundary in about one case of sqrt(dk): 2e-3 of the outputs.  States that keep 17 bits
    give 3e-3 (the plain op) to 8e-3 here.  (Of the gradients only dv of a POP call with
    whole chunks per block: there both sides weigh the same operand of the same chunks.)"""
    choose_backward(PASSES)
    decays = (0.97,)
    q, k, v, s = hp.make_inputs(1, T, 1, dk, dv, seed=T + block, state_std=0.5)
    if block:
        d_o, d_b = hp.make_cotangents([(1, T, 1, dv), (1, T // block, 1, dk, dv)], seed=T)
        n = emu_lib.fp_pop_retention_workspace_bytes(1, T, 1, dk, dv, block)
        ws, p = torch.empty(n, dtype=torch.uint8), hp._p
        o, states, (dq, dk_, dv_) = torch.empty_like(v), torch.empty_like(d_b), [torch.empty_like(t) for t in (q, k, v)]
        assert n > 0 and emu_lib.fp_pop_retention_fwd_split(p(q), p(k), p(v), p(s), hp._dec(decays), p(o), p(states), 1, T, 1, dk, dv, block,
                                                            p(ws), n, None) == 0
        assert emu_lib.fp_pop_retention_bwd_split(p(q), p(k), p(v), p(s), hp._dec(decays), p(d_o), p(d_b), p(dq), p(dk_), p(dv_), None,
                                                  1, T, 1, dk, dv, block, p(ws), n, 1, None) == 0
        pairs = [("o", o, hp.raw_pop_fwd(emu_lib, q, k, v, s, decays, block)[0]),
                 ("dv", dv_, hp.raw_pop_bwd(emu_lib, q, k, v, s, decays, block, d_o, d_b)[2])]
    else:
        o, _, n = hp.raw_split_fwd(emu_lib, q, k, v, s, decays)
        assert n > 0
        pairs = [("o", o, hp.raw_fwd(emu_lib, q, k, v, s, decays)[0])]
    for name, cut, uncut in pairs:
        share = (cut != uncut).float().mean().item()
        print(name, share)
        assert share <= 2e-3, (name, share)


@pytest.mark.parametrize("T,dk,dv", [
    (511, 128, 128),    # the 128-wide state-only kernel, a last chunk of 63 tokens
    (257, 128, 256),    # of one token, two workgroups per segment
    (330, 64, 128),     # 64-row states, a last chunk of 10 tokens
])
def test_cut_final_state_follows_the_uncut_walk(emu_lib, T, dk, dv):
    """The state-only walk of a cut call takes the chunks of the uncut one, the short one last, and weighs the same keys the
    same way, so that the final state (bf16 of an fp32 sum, see above: half a step in 2^13 or so) is the uncut one's."""
    q, k, v, s = hp.make_inputs(1, T, 1, dk, dv, seed=T, state_std=0.5)
    _, S, n = hp.raw_split_fwd(emu_lib, q, k, v, s, (0.97,))
    _, S1 = hp.raw_fwd(emu_lib, q, k, v, s, (0.97,))
    share = (S != S1).float().mean().item()
    assert n > 0 and share <= 1e-3, share


@pytest.mark.parametrize("reverse", (0, 1))
@pytest.mark.parametrize("T,total,dk,dv", [
    (144, 360, 64, 64),     # a short chunk in every segment, the last one shorter still
    (128, 257, 64, 192),    # whole chunks, a last segment of one token; three workgroups per segment
    (63, 63, 64, 64),       # less than a chunk
])
def test_state_only_kernel_matches_the_walk(emu_lib, T, total, dk, dv, reverse):
    """Where the state-only kernel takes 64-row states it cuts the chunks, weighs the operands and sums as the pass kernel's
    state-only walk does, in either direction: same bits."""
    segs, H = -(-total // T), 2
    w, _, z, _ = hp.make_inputs(1, total, H, dk, dv, seed=T + dv)
    out = []
    for walk in (0, 1):
        u = torch.zeros(2, segs, H, dk, dv, dtype=torch.int16)
        rc = emu_lib.emu_state_only(walk, hp._p(w), hp._p(z), hp._p(u[0]), hp._p(u[1]), segs, T, H, dk, dv,
                                    segs, total, reverse, ctypes.c_float(-0.03))
        assert rc == 0
        out.append(u)
    assert out[0].any() and torch.equal(out[0], out[1])


def test_rule_of_the_state_only_pass(emu_lib):
    """Which kernel sums the segments of a cut call, at 256 units: of 64-row states the state-only kernel but for many workgroups
    of short segments (4 096 of a chunk: 28 us in the walk, 34 in the kernel); the walk for all other states but those of 128 x 128."""
    pays = emu_lib.emu_contrib_pays
    assert pays(1, 64, 1, 64, 64, 256) and pays(32, 1000, 4, 64, 128, 256) and pays(96, 64, 4, 64, 128, 256)
    assert not pays(97, 256, 4, 64, 128, 256) and pays(97, 257, 4, 64, 128, 256) and pays(4096, 257, 4, 64, 64, 256)
    assert not pays(97, 1000, 8, 128, 64, 256) and not pays(108, 128, 12, 128, 64, 256) and not pays(97, 1000, 4, 128, 192, 256)
    assert pays(1, 64, 1, 128, 128, 256) and pays(1000, 64, 8, 128, 256, 256)


@pytest.mark.parametrize("T,dk,dv", [
    (257, 64, 64),      # 64-row states: a last segment of one token
    (575, 64, 192),     # ... three workgroups per segment, a last chunk of 63 tokens
    (513, 128, 64),     # 128-row states, 64 columns per workgroup (the walk)
    (577, 128, 192),    # ... a last segment of one token (uneven cuts all: equal segments hand bf16 states on, a step in 2^8)
])
def test_state_only_pass_in_64_columns(emu_lib, T, dk, dv):
    """What the segments add to the carried state, 64 columns per workgroup: the final state is the uncut call's (up to the half
    step in 2^13 of test_cut_final_state_follows_the_uncut_walk; gamma = 0.97 over the last 64 tokens: the short chunk counts),
    and the gradient of the initial state, which the walk back gives, meets the oracle."""
    q, k, v, s = hp.make_inputs(1, T, 1, dk, dv, seed=T, state_std=0.5)
    d_o, d_s = hp.make_cotangents([(1, T, 1, dv), (1, 1, dk, dv)], seed=T + 1)
    o, S, n = hp.raw_split_fwd(emu_lib, q, k, v, s, (0.97,))
    _, S1 = hp.raw_fwd(emu_lib, q, k, v, s, (0.97,))
    assert n > 0 and (S != S1).float().mean().item() <= 1e-3
    o_ref, _, (_, _, _, gs) = hp.oracle_plain(q, k, v, s, (0.97,), d_o, d_s)
    ds0 = hp.raw_split_bwd(emu_lib, q, k, v, s, (0.97,), d_o, d_s)[3]
    _check_all([("o", o, o_ref), ("ds0", ds0, gs)])


@pytest.mark.parametrize("B,nblk,block,Ls,H,state_std,dk,dv", [
    (1, 2, 128, 16, 1, 0.5, 128, 128),     # two chunks per block
    (1, 4, 64, 64, 1, None, 128, 128),     # block == chunk, suffixes as long as a chunk, no initial state
    (1, 1, 192, 1, 2, 0.3, 128, 128),      # three chunks per block, one-token suffixes, two heads
    (1, 8, 64, 9, 1, 0.3, 128, 128),       # short suffixes folded into every chunk; 9 suffixes over 3 workgroups of the second kernel
    (1, 4, 64, 16, 2, 0.3, 64, 128),       # 64-wide keys: folded suffixes
    (1, 2, 128, 40, 1, None, 128, 64),     # 64-wide values: suffixes as stops, no initial state
    (1, 4, 64, 9, 1, 0.5, 64, 64),         # 64 x 64 states: four state tiles for eight waves
])
def test_fused_pop_backward_that_carries_ds_once(emu_lib, choose_backward, B, nblk, block, Ls, H, state_std, dk, dv):
    """dk, dv of 64 or 128, whole chunks per block (forced here at lengths below the eight chunks from which the
    library chooses it by itself): the fused POP backward runs in
    the kernel that walks backward once for dk and dv beside a forward walk for dq, with the
    suffixes as extra stops at the block boundaries or folded into the chunks there.  Same results as the
    pass-per-gradient path."""
    decays = oracle.head_decays(H, (4, 9))
    T = nblk * block
    q, k, v, s = hp.make_inputs(B, T, H, dk, dv, seed=T + Ls, state_std=state_std)
    sfx = hp.make_suffix_inputs(B, nblk, Ls, H, dk, dv, seed=T + Ls + 1)
    cot = hp.make_cotangents([(B, T, H, dv), tuple(sfx[2].shape), (B, H, dk, dv)], seed=T + 2)
    choose_backward(FUSED)
    grads = hp.raw_fused_bwd(emu_lib, q, k, v, s, sfx, decays, block, cot)
    _, _, _, g_ref = hp.oracle_fused(q, k, v, s, sfx, decays, block, cot)
    _check_all([(n, g, r) for n, g, r in zip(FUSED_NAMES, grads, g_ref)])
    choose_backward(PASSES)
    other = hp.raw_fused_bwd(emu_lib, q, k, v, s, sfx, decays, block, cot)
    differs = False
    for name, x, y in zip(FUSED_NAMES, grads, other):
        if x is not None:
            assert hp.error_report(x, y.float())["rms_ratio"] < 0.004, name
            differs = differs or not torch.equal(x, y)
    assert differs, "the forced choice made no difference: both calls took the same kernels"


@pytest.mark.parametrize("B,T,H,state_std,every,dk,dv", [
    (1, 330, 1, 0.5, 128, 128, 128),      # ragged tail beyond the last checkpoint, initial state
    (1, 256, 1, None, 128, 128, 128),     # the sequence ends on a checkpoint, no initial state
    (2, 200, 1, 0.3, 64, 128, 128),       # a checkpoint after every chunk, two sequences
    (1, 200, 1, 0.2, 1024, 128, 128),     # interval longer than the sequence: no checkpoint at all
    (1, 260, 1, 0.4, 0, 128, 128),        # no checkpoint buffer: the fused backward walks forward from s0
    (1, 330, 2, 0.5, 128, 64, 128),       # 64-wide keys
    (1, 210, 1, None, 0, 128, 64),        # 64-wide values, no checkpoints, no initial state
    (1, 300, 1, 0.3, 128, 64, 64),        # 64 x 64 states
    (1, 330, 2, 0.5, -128, 128, 128),     # the two workgroups of a stream paced (the harness runs them in turn: no waiting)
])
def test_fused_backward_with_checkpoints(emu_lib, choose_backward, B, T, H, state_std, every, dk, dv):
    """dk, dv of 64 or 128 (forced here at lengths below the eight chunks from which the library chooses it by
    itself): the backward that carries dS once, beside the
    workgroup that re-runs the state from the checkpoints the forward left (segments taken from
    the last to the first)."""
    choose_backward(PACED if every < 0 else FUSED)
    every = abs(every)
    decays = oracle.head_decays(H)
    q, k, v, s = hp.make_inputs(B, T, H, dk, dv, seed=T, state_std=state_std)
    d_o, d_s = hp.make_cotangents([(B, T, H, dv), (B, H, dk, dv)], seed=T + 1)
    if every:
        o, S, dq, dk_, dv_, ds0 = hp.raw_ckpt_fwd_bwd(emu_lib, q, k, v, s, decays, d_o, d_s, every)
    else:
        o, S = hp.raw_fwd(emu_lib, q, k, v, s, decays)
        dq, dk_, dv_, ds0 = hp.raw_bwd(emu_lib, q, k, v, s, decays, d_o, d_s)
    o_ref, S_ref, (gq, gk, gv, gs) = hp.oracle_plain(q, k, v, s, decays, d_o, d_s)
    _check_all([("o", o, o_ref), ("S", S, S_ref), ("dq", dq, gq), ("dk", dk_, gk), ("dv", dv_, gv), ("ds0", ds0, gs)])
    # the checkpoints only serve dq: everything else is bit for bit what the entry points without them give
    o2, S2 = hp.raw_fwd(emu_lib, q, k, v, s, decays)
    g2 = hp.raw_bwd(emu_lib, q, k, v, s, decays, d_o, d_s)
    assert torch.equal(o, o2) and torch.equal(S, S2)
    assert torch.equal(dk_, g2[1]) and torch.equal(dv_, g2[2])
    assert (ds0 is None and g2[3] is None) or torch.equal(ds0, g2[3])
    # and the pass-per-gradient backward gives other bits: the forced choice is what ran
    choose_backward(PASSES)
    g3 = hp.raw_bwd(emu_lib, q, k, v, s, decays, d_o, d_s)
    assert not torch.equal(g3[1], dk_)


@pytest.mark.parametrize("B,T,H,dk,dv,state_std,want_ds0", [
    (5, 16, 2, 128, 128, 0.5, True),     # more (sequence, head) pairs than the harness runs workgroups
    (7, 31, 1, 64, 128, 0.5, True),      # two k-steps along the tokens, 64-wide keys
    (3, 9, 2, 128, 64, None, True),      # no state: no read-out, no d_s0
    (4, 32, 1, 64, 64, 0.3, True),       # the longest sequence the kernel takes
    (2, 1, 3, 128, 128, 0.5, True),      # one token
    (3, 17, 2, 64, 128, 0.5, False),     # d_s0 not wanted
])
def test_many_short_sequences(emu_lib, choose_backward, B, T, H, dk, dv, state_std, want_ds0):
    """At most 32 tokens per sequence, a state per sequence (the suffix call of the reference's POP layer): forward
    and, with no gradient of the final state, backward take one (sequence, head) pair per step in kernels of their
    own."""
    decays = oracle.head_decays(H, (4, 9))
    q, k, v, s = hp.make_inputs(B, T, H, dk, dv, seed=T + dk, state_std=state_std)
    d_o, = hp.make_cotangents([(B, T, H, dv)], seed=T + 1)
    o, S = hp.raw_fwd(emu_lib, q, k, v, s, decays)
    o_only, none = hp.raw_fwd(emu_lib, q, k, v, s, decays, want_state=False)
    grads = hp.raw_bwd(emu_lib, q, k, v, s, decays, d_o, None, want_ds0=want_ds0)
    o_ref, S_ref, ref = hp.oracle_plain(q, k, v, s, decays, d_o, None)
    _check_all([("o", o, o_ref), ("S", S, S_ref)])
    assert none is None and torch.equal(o_only, o)
    _check_all([(n, g, r) for n, g, r in zip(("dq", "dk", "dv", "ds0"), grads, ref) if g is not None])
    choose_backward(PASSES)
    o_p, S_p = hp.raw_fwd(emu_lib, q, k, v, s, decays)
    assert not torch.equal(S_p, S), "the forced choice made no difference: both forwards took the same kernel"
    assert hp.error_report(o, o_p.float())["rms_ratio"] < 0.004 and hp.error_report(S, S_p.float())["rms_ratio"] < 0.006
    other = hp.raw_bwd(emu_lib, q, k, v, s, decays, d_o, None, want_ds0=want_ds0)
    for n, x, y in zip(("dq", "dk", "dv", "ds0"), grads, other):
        if x is not None:
            assert hp.error_report(x, y.float())["rms_ratio"] < 0.004, n
    # with a gradient of the final state the chunk kernels run, and give the same dq (the short kernel's only
    # state term) up to the rounding of its partial sums
    d_s, = hp.make_cotangents([(B, H, dk, dv)], seed=T + 2)
    choose_backward(0)
    with_ds = hp.raw_bwd(emu_lib, q, k, v, s, decays, d_o, d_s, want_ds0=want_ds0)
    _, _, ref_ds = hp.oracle_plain(q, k, v, s, decays, d_o, d_s)
    _check_all([(n, g, r) for n, g, r in zip(("dq", "dk", "dv", "ds0"), with_ds, ref_ds) if g is not None])


def test_c_entry_points_refuse_a_capturing_stream(emu_lib):
    """The entry points that launch the pass kernels return FP_ERR_LAUNCH, before launching anything, when
    their stream is recording a HIP graph (the harness's stand-in for hipStreamIsCapturing is a flag);
    the decode step stays capturable."""
    import ctypes
    decays = oracle.head_decays(1)
    q, k, v, s = hp.make_inputs(1, 70, 1, 64, 64, seed=1, state_std=0.5)
    d_o, = hp.make_cotangents([(1, 70, 1, 64)], seed=2)
    sfx = hp.make_suffix_inputs(1, 1, 8, 1, 64, 64, seed=3)
    cot = hp.make_cotangents([(1, 70, 1, 64), tuple(sfx[2].shape), (1, 1, 64, 64)], seed=4)
    calls = [
        lambda: hp.raw_fwd(emu_lib, q, k, v, s, decays),
        lambda: hp.raw_bwd(emu_lib, q, k, v, s, decays, d_o, None),
        lambda: hp.raw_pop_fwd(emu_lib, q, k, v, s, decays, 32),
        lambda: hp.raw_pop_bwd(emu_lib, q, k, v, s, decays, 32, d_o, None),
        lambda: hp.raw_fused_fwd(emu_lib, q, k, v, s, sfx, decays, 64),
        lambda: hp.raw_fused_bwd(emu_lib, q, k, v, s, sfx, decays, 64, cot),
        lambda: hp.raw_split_fwd(emu_lib, q, k, v, s, decays),
        lambda: hp.raw_split_bwd(emu_lib, q, k, v, s, decays, d_o, None),
        lambda: hp.raw_ckpt_fwd_bwd(emu_lib, q, k, v, s, decays, d_o, None, 64),
    ]
    emu_lib.emu_set_capturing(1)
    try:
        for call in calls:
            with pytest.raises(AssertionError, match="rc=-5: .*capturing a HIP graph"):
                call()
        o = torch.zeros(1, 70, 1, 64, dtype=hp.BF16)
        rc = emu_lib.fp_retention_fwd_split_static(hp._p(q), hp._p(k), hp._p(v), hp._p(s), hp._dec(decays), hp._p(o), None,
                                                  1, 70, 1, 64, 64, None)
        assert rc == -5 and b"capturing" in emu_lib.fp_last_error()
        hp.raw_decode_step(emu_lib, q[:, 0], k[:, 0], v[:, 0], s, decays)
    finally:
        emu_lib.emu_set_capturing(0)
    hp.raw_fwd(emu_lib, q, k, v, s, decays)


def test_checkpoint_size_query(emu_lib, choose_backward):
    """fp_retention_checkpoint_bytes: 0 where the fused backward would not run or the sequence is
    no longer than one interval, else B * (T / every) state matrices."""
    import ctypes
    every = ctypes.c_int(-1)
    choose_backward(FUSED)
    assert emu_lib.fp_retention_checkpoint_bytes(2, 4096, 4, 128, 128, ctypes.byref(every)) == 2 * 2 * (4096 // 512) * 4 * 128 * 128
    assert every.value == 512
    assert emu_lib.fp_retention_checkpoint_bytes(2, 512, 4, 128, 128, ctypes.byref(every)) == 0 and every.value == 0
    assert emu_lib.fp_retention_checkpoint_bytes(2, 4096, 4, 64, 128, ctypes.byref(every)) == 2 * 2 * (4096 // 512) * 4 * 64 * 128
    assert emu_lib.fp_retention_checkpoint_bytes(2, 4096, 4, 64, 256, ctypes.byref(every)) == 0
    assert emu_lib.fp_retention_checkpoint_bytes(2, 4096, 4, 128, 128, None) > 0
    choose_backward(PASSES)
    assert emu_lib.fp_retention_checkpoint_bytes(2, 4096, 4, 128, 128, ctypes.byref(every)) == 0


@pytest.mark.parametrize("B,H,dk,dv", [(2, 3, 64, 128), (1, 2, 128, 64), (1, 1, 256, 256), (1, 2, 192, 192), (2, 1, 64, 192),
                                       (1, 130, 64, 64)])   # more than 128 heads
def test_decode_step(emu_lib, B, H, dk, dv):
    """Three chained steps (no state, fresh buffer, in place) against the oracle's recurrent step."""
    decays = oracle.head_decays(H)
    g = torch.Generator().manual_seed(dk + dv)
    state, ref_state = None, None
    for step in range(3):
        q, k = (torch.randn(B, H, dk, generator=g).to(hp.BF16) for _ in range(2))
        v = torch.randn(B, H, dv, generator=g).to(hp.BF16)
        o, state = hp.raw_decode_step(emu_lib, q, k, v, state, decays, in_place=step == 2)
        o_ref, ref_state = oracle.recurrent_step(q.float(), k.float(), v.float(), ref_state, decays)
        hp.assert_close(o, o_ref, f"o step {step}")
        hp.assert_close(state, ref_state, f"state step {step}")
        ref_state = state.float()    # follow the kernel's bf16 state, as a decode loop does


def test_optional_outputs_and_determinism(emu_lib):
    decays = oracle.head_decays(2)
    q, k, v, s = hp.make_inputs(1, 90, 2, 64, 64, seed=3, state_std=0.5)
    o1, S1 = hp.raw_fwd(emu_lib, q, k, v, s, decays)
    o2, none = hp.raw_fwd(emu_lib, q, k, v, s, decays, want_state=False)
    assert none is None and torch.equal(o1, o2)
    d_o, = hp.make_cotangents([(1, 90, 2, 64)], seed=4)
    g1 = hp.raw_bwd(emu_lib, q, k, v, s, decays, d_o, None)
    g2 = hp.raw_bwd(emu_lib, q, k, v, s, decays, d_o, None, want_ds0=False)
    assert g2[3] is None and all(torch.equal(a, b) for a, b in zip(g1[:3], g2[:3]))
    z = torch.zeros(1, 2, 64, 64, dtype=hp.BF16)
    g3 = hp.raw_bwd(emu_lib, q, k, v, s, decays, d_o, z)
    assert all(torch.equal(a, b) for a, b in zip(g1, g3))


def test_gamma_one_and_tiny(emu_lib):
    """gamma = 1 (no decay) and a gamma small enough that gamma^63 underflows."""
    decays = (1.0, 1e-3)
    q, k, v, s = hp.make_inputs(1, 130, 2, 64, 64, seed=9, state_std=0.5)
    o, S = hp.raw_fwd(emu_lib, q, k, v, s, decays)
    o_ref, S_ref = hp.oracle_plain(q, k, v, s, decays)
    hp.assert_close(o, o_ref, "o")
    hp.assert_close(S, S_ref, "S")


@pytest.mark.parametrize("B,T,H,d,vec", [(2, 37, 3, 64, False), (3, 5, 2, 128, True), (1, 300, 1, 8, False),
                                         (1, 4096, 5, 64, False)])   # enough tokens for one thread to take all heads
def test_rotary(emu_lib, B, T, H, d, vec):
    """Rotation of q and k (also q alone, in place, and back) against the oracle."""
    g = torch.Generator().manual_seed(d + T)
    q, k = (torch.randn(B, T, H, d, generator=g).to(hp.BF16) for _ in range(2))
    theta = oracle.position_thetas(d)
    start = torch.tensor([7, 4000, 123456][:B]) if vec else 1000
    pos = (start[:, None] if vec else start) + torch.arange(T)[None]
    rq, rk = hp.raw_rotary(emu_lib, q, k, theta, start)

    def same(got, ref):
        """Equal, or (libm's and torch's sine may differ in the last place of an fp32 angle of a few
        thousand radians) a handful of elements apart by one bf16 step."""
        diff = (got.float() - ref.float()).abs()
        return bool((diff > 0).float().mean() < 1e-4) and bool((diff <= ref.float().abs() * 2.0 ** -7 + 1e-5).all())

    assert same(rq, oracle.rotary(q, pos, theta)) and same(rk, oracle.rotary(k, pos, theta))
    only_q, none = hp.raw_rotary(emu_lib, q, None, theta, start)
    assert none is None and torch.equal(only_q, rq)
    back_q, back_k = hp.raw_rotary(emu_lib, rq, rk, theta, start, inverse=True)
    assert same(back_q, oracle.rotary(rq, pos, theta, inverse=True))
    hp.assert_close(back_k, k.float(), "round trip")
    q2, k2 = q.clone(), k.clone()
    hp.raw_rotary(emu_lib, q2, k2, theta, start, in_place=True)
    assert torch.equal(q2, rq) and torch.equal(k2, rk)


@pytest.mark.parametrize("rows,H,dv", [(19, 3, 64), (5, 2, 128), (3, 1, 256), (70, 5, 8)])
def test_gated_group_norm(emu_lib, rows, H, dv):
    g = torch.Generator().manual_seed(rows + dv)
    r = (torch.randn(rows, H, dv, generator=g) * 2 + 0.5).to(hp.BF16)
    gate = torch.randn(rows, H * dv, generator=g).to(hp.BF16)
    d_out = torch.randn(rows, H * dv, generator=g).to(hp.BF16)
    out = hp.raw_gated_norm_fwd(emu_lib, r, gate)
    ref = oracle.gated_group_norm(r, gate)
    # same rounding points as the oracle: equal except where an fp32 value sits on a bf16 rounding boundary
    differ = (out.float() - ref.float()).abs()
    assert float((differ > 0).float().mean()) < 0.01, float((differ > 0).float().mean())
    hp.assert_close(out, ref.float(), "out")
    d_r, d_g = hp.raw_gated_norm_bwd(emu_lib, r, gate, d_out)
    d_r_ref, d_g_ref = hp.oracle_gated_norm_grads(r, gate, d_out)
    hp.assert_close(d_r, d_r_ref, "d_r")
    hp.assert_close(d_g, d_g_ref, "d_g")


@pytest.mark.parametrize("B,T,state_std", [
    (1, 33, 0.5), (1, 64, None), (1, 65, 0.5), (2, 128, 0.5), (1, 193, 0.5), (1, 257, None),   # one chunk to five: fewer than are under way, and more
    (17, 64, 0.5), (18, 65, 0.5), (17, 129, 0.5),   # several sequences per workgroup (8 units), of one chunk to three
])
def test_pass_of_64_wide_rows(emu_lib, choose_backward, B, T, state_std):
    """The pass whose rows are copied straight into LDS, in all four roles: forward and the three gradient passes."""
    choose_backward(PASSES)
    test_plain_fwd_bwd(emu_lib, B, T, 1, 64, 64, state_std)


def test_pass_of_64_wide_rows_fp32_states_every_chunk(emu_lib):
    """Segments of one chunk with fp32 states, several per workgroup: a state's two tiles are taken in turn by three chunks in a row."""
    test_pop_split_at_blocks(emu_lib, 1, 1300, 1, 64, 64, 64, 0.5, 21)


def test_pass_of_64_wide_rows_fp32_states_every_second_chunk(emu_lib):
    """... of two chunks: the state of a chunk is asked for in the step that carries the last one that brought its own."""
    test_pop_split_at_blocks(emu_lib, 1, 1300, 1, 64, 64, 128, 0.5, 11)


@pytest.mark.parametrize("late", [256, -256], ids=["carry", "others"])
def test_copies_do_not_overtake_what_reads_them(emu_lib, choose_backward, late):
    """The waves that carry the state (the first four) come late out of every barrier, or all others do: nothing is copied, scored, weighed
    or stored over what a wave of the same step still reads."""
    emu_lib.emu_set_lag(late, 3000)
    try:
        test_pop_split_at_blocks(emu_lib, 1, 2304, 1, 64, 64, 64, 0.5, 36)   # five fp32 states in a row for half of the workgroups
        test_folded_forward(emu_lib, 1, 6, 65, 16, 1, 64, 0.5)
        choose_backward(PASSES)
        test_pass_of_128_columns_per_workgroup(emu_lib, choose_backward, 5, 300, 1, 128, 0.5)
    finally:
        emu_lib.emu_set_lag(0, 0)


@pytest.mark.parametrize("T,block", [(192, 64), (300, 64), (200, 40), (260, 130)])
def test_pass_of_64_wide_rows_blocks(emu_lib, choose_backward, T, block):
    """Block states leave, and their gradients join, at every chunk and at some of them."""
    choose_backward(PASSES)
    test_pop_fwd_bwd(emu_lib, 1, T, 1, 64, 64, block)


@pytest.mark.parametrize("B,T,H,dv,state_std", [
    (5, 33, 1, 128, 0.5), (5, 64, 1, 128, None), (3, 65, 1, 256, 0.5), (5, 96, 1, 128, 0.5),   # fewer halves of chunks than are under way
    (5, 161, 1, 128, 0.5), (2, 200, 2, 256, None), (5, 257, 1, 128, 0.5),                        # more
    (9, 400, 1, 128, 0.5),                                                                       # more workgroups than units (8)
])
def test_pass_of_128_columns_per_workgroup(emu_lib, choose_backward, B, T, H, dv, state_std):
    """The pass with 128 columns per workgroup and half a chunk per step, in the roles that it has: forward and dv pass, with values of
    128 the dq and dk passes (which share a launch with it)."""
    assert emu_lib.emu_pass_kernel(1, B, T, H, 128, dv, 0, 0, 0, 8) == WIDE
    choose_backward(PASSES)
    test_plain_fwd_bwd(emu_lib, B, T, H, 128, dv, state_std)


@pytest.mark.parametrize("B,T,dv,block", [
    (6, 256, 128, 64),     # a block state behind every chunk
    (3, 320, 256, 128),    # two column blocks per workgroup, tokens after the last boundary
])
def test_outputs_do_not_depend_on_block_states(emu_lib, B, T, dv, block):
    """128-wide keys on more than half of the units: the plain forward runs in the kernel with 128 columns per workgroup, one that leaves
    block states (POP, checkpoints) in the one with 64.  o is the same bit for bit, and so is the state after the last token."""
    decays = oracle.head_decays(1, (4, 9))
    q, k, v, s = hp.make_inputs(B, T, 1, 128, dv, seed=T + dv, state_std=0.5)
    o, S = hp.raw_fwd(emu_lib, q, k, v, s, decays)
    o_pop, states = hp.raw_pop_fwd(emu_lib, q, k, v, s, decays, block)
    assert torch.equal(o, o_pop)
    assert T % block != 0 or torch.equal(S, states[:, -1])
    if dv == 128:
        d_o, d_s = hp.make_cotangents([(B, T, 1, dv), (B, 1, 128, dv)], seed=T)
        o_ckpt, S_ckpt = hp.raw_ckpt_fwd_bwd(emu_lib, q, k, v, s, decays, d_o, d_s, 128)[:2]
        assert torch.equal(o, o_ckpt) and torch.equal(S, S_ckpt)


def _shifted(t):
    """The same values two bytes behind where they would be aligned."""
    if t is None:
        return None
    flat = torch.empty(t.numel() + 1, dtype=t.dtype)
    flat[1:] = t.flatten()
    assert flat[1:].data_ptr() % 4 == 2
    return flat[1:].view(t.shape)


@pytest.mark.parametrize("which,B,T,dk,dv,block,Ls", [
    *[(which, 1, 100, 64, 64, 0, 0) for which in ("q", "k", "v", "s", "all")],   # one sequence per workgroup
    *[(which, 9, 40, 64, 128, 0, 0) for which in ("k", "all")],                  # several
    *[(which, 1, 150, 64, 64, 64, 0) for which in ("v", "s", "all")],            # block states
    *[(which, 1, 128, 64, 64, 64, 16) for which in ("q", "s", "sfx", "all")],    # folded suffixes
    *[(which, 6, 100, 128, 128, 0, 0) for which in ("q", "all")],                # 128 columns per workgroup
])
def test_tensors_that_are_not_aligned(emu_lib, choose_backward, which, B, T, dk, dv, block, Ls):
    """Tensors at any address are taken, as by loads into registers, and none is copied straight into LDS from one that is no multiple of
    16 bytes, for which such copies are not made."""
    choose_backward(PASSES)
    decays = oracle.head_decays(1, (4, 9))
    q, k, v, s = hp.make_inputs(B, T, 1, dk, dv, seed=T, state_std=0.5)
    move = lambda name, t: _shifted(t) if which in (name, "all") else t
    ins = [move(name, t) for name, t in zip("qkvs", (q, k, v, s))]
    emu_lib.emu_misaligned_fills()
    if Ls:
        sfx = hp.make_suffix_inputs(B, T // block, Ls, 1, dk, dv, seed=T + 1)
        got = hp.raw_fused_fwd(emu_lib, *ins, [move("sfx", t) for t in sfx], decays, block)
        ref = hp.oracle_fused(q, k, v, s, sfx, decays, block)
    elif block:
        d_o, d_b = hp.make_cotangents([(B, T, 1, dv), (B, T // block, 1, dk, dv)], seed=T)
        got = hp.raw_pop_fwd(emu_lib, *ins, decays, block) + hp.raw_pop_bwd(emu_lib, *ins, decays, block, move("v", d_o), move("s", d_b))
        o_ref, st_ref, grads = hp.oracle_pop(q, k, v, s, decays, block, d_o, d_b)
        ref = (o_ref, st_ref, *grads)
    else:
        d_o, d_s = hp.make_cotangents([(B, T, 1, dv), (B, 1, dk, dv)], seed=T)
        got = hp.raw_fwd(emu_lib, *ins, decays) + hp.raw_bwd(emu_lib, *ins, decays, move("v", d_o), move("s", d_s))
        o_ref, S_ref, grads = hp.oracle_plain(q, k, v, s, decays, d_o, d_s)
        ref = (o_ref, S_ref, *grads)
    assert emu_lib.emu_misaligned_fills() == 0
    for i, (g, r) in enumerate(zip(got, ref)):
        hp.assert_close(g, r, f"output {i}")


@pytest.mark.parametrize("B,T,dk,dv,block", [
    (1, 200, 64, 64, 0), (2, 130, 64, 128, 0),    # one sequence per workgroup
    (20, 64, 64, 64, 0), (9, 100, 64, 128, 0),    # several
    (1, 200, 64, 128, 64), (2, 130, 64, 64, 50),  # block states
    (6, 200, 128, 128, 0), (3, 130, 128, 256, 0),  # 128 columns per workgroup: outputs and states (its walk backward adds half chunks in turn)
])
def test_outputs_do_not_depend_on_alignment(emu_lib, choose_backward, B, T, dk, dv, block):
    """Aligned tensors are copied straight into LDS, others go through registers in another kernel, which a rule may choose for aligned ones,
    too: outputs, states and gradients are the same bit for bit."""
    choose_backward(PASSES)
    decays = oracle.head_decays(1, (4, 9))
    q, k, v, s = hp.make_inputs(B, T, 1, dk, dv, seed=T + B, state_std=0.5)
    d_o, d_s = hp.make_cotangents([(B, T, 1, dv), (B, T // block, 1, dk, dv) if block else (B, 1, dk, dv)], seed=T)

    def outputs(move):
        q_, k_, v_, s_, do_, ds_ = (move(t) for t in (q, k, v, s, d_o, d_s))
        if block:
            return hp.raw_pop_fwd(emu_lib, q_, k_, v_, s_, decays, block) + hp.raw_pop_bwd(emu_lib, q_, k_, v_, s_, decays, block, do_, ds_)
        forward = hp.raw_fwd(emu_lib, q_, k_, v_, s_, decays)
        return forward if dk == 128 else forward + hp.raw_bwd(emu_lib, q_, k_, v_, s_, decays, do_, ds_)

    for i, (a, b) in enumerate(zip(outputs(lambda t: t), outputs(_shifted))):
        assert torch.equal(a, b), f"output {i}: {(a != b).sum().item()} elements differ"


@pytest.mark.parametrize("kernel,passes,B,T,H,dv", [
    (4, 1, 256, 64, 1, 64),       # one workgroup per sequence while they fit the device at once
    (25, 1, 257, 64, 1, 64),
    (25, 1, 43, 33, 12, 128),
    (25, 1, 96, 1, 8, 128),
    (3, 1, 97, 64, 8, 128),       # more than six per unit
    (25, 1, 24, 64, 16, 256),
    (3, 1, 257, 65, 1, 64),       # a second chunk
    (3, 2, 257, 64, 1, 64),       # passes that share a launch
])
def test_rule_of_sequences_of_one_chunk(emu_lib, kernel, passes, B, T, H, dv):
    """Which forwards of 64-wide keys and at most one chunk go through registers, at 256 units."""
    assert emu_lib.emu_pass_kernel(passes, B, T, H, 64, dv, 0, 0, 0, 256) == kernel


@pytest.mark.parametrize("B,T,dv", [(9, 64, 64), (48, 64, 64), (49, 40, 64), (13, 33, 128), (5, 50, 256)])
def test_sequences_of_one_chunk(emu_lib, B, T, dv):
    """Forwards of short sequences on more workgroups than the device has units (8), on both sides of the rule."""
    assert (emu_lib.emu_pass_kernel(1, B, T, 1, 64, dv, 0, 0, 0, 8) == 25) == (B * dv // 64 <= 48)
    decays = oracle.head_decays(1, (4, 9))
    q, k, v, s = hp.make_inputs(B, T, 1, 64, dv, seed=T, state_std=0.5)
    (o, S), (o_ref, S_ref) = hp.raw_fwd(emu_lib, q, k, v, s, decays), hp.oracle_plain(q, k, v, s, decays)
    _check_all([("o", o, o_ref), ("s_out", S, S_ref)])
