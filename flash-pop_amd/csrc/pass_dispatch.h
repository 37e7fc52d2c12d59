// Validation of one pass launch and the choice of kernel instantiation, shared by the device
// launcher and the CPU thread harness so that both take the same decisions.
#pragma once
#include <cstring>
#include <initializer_list>

#include "pass_args.h"
#include "retention_pass_ws.h"
#include "retention_pass_fill.h"
#include "retention_pass_wide.h"

namespace fpk {

// Number of kernel instantiations `dispatch_pass` can pick from (its `slot` argument is below this).
constexpr int PASS_KERNELS = 27;
constexpr int FILL_SLOTS = 5;   // those of retention_pass_fill.h that walk either way are below this

// Checks what the walks assume about `a` and chooses a.slots (workgroups per (head, column tile))
// for a device with `compute_units` units.  Returns nullptr, or a message for the caller.
inline const char* plan_pass(PassArgs& a, int compute_units) {
  const bool blocks = a.block > 0 && (a.Bout || a.Bin);
  const bool narrow = a.dA == 64 || a.dA == 128;   // one visit per chunk
  const bool suffix = a.Ls > 0;
  if (a.segs < 0 || (a.segs > 0 && (blocks || suffix || a.B % a.segs != 0 || a.total > (long long)a.segs * a.T ||
                                    a.total <= (a.segs - 1LL) * a.T)))
    return "segments that do not cover their sequence, or segments with block states or suffixes";
  if ((a.R0lo && (!a.R0 || blocks || suffix)) || (a.Rout_lo && (!a.Rout || !a.state_only)))
    return "fp32 states that this walk does not take";
  if (a.dA != 64 && a.dA != 128 && a.dA != 192 && a.dA != 256) return "unsupported contraction width (dA must be 64, 128, 192 or 256)";
  if (a.dB < BV || a.dB % BV != 0) return "dB must be a multiple of 64";
  if (suffix) {
    // the C-ABI layer reports these to the caller in its own words
    if (blocks || a.block <= 0 || a.nblk != a.T / a.block || !a.Xs || !a.Ws || !a.Zs || !a.Ys)
      return "suffix walk: needs nblk == T / block and all four suffix tensors";
    if (a.Ls > CH && !narrow) return "suffixes longer than 64 tokens need dk and dv of 64 or 128";
    a.slots = a.B;
  }
  // One workgroup per (batch entry, head, column tile) while that fits the chip once; beyond that
  // the plain walk lets each workgroup take several batch entries one after another, which keeps
  // its load pipeline full across short sequences.
  if (a.slots <= 0) {
    a.slots = a.B;
    if (narrow && !blocks && !suffix) {
      int fit = compute_units / (a.H * (a.dB / BV));
      if (fit < 1) fit = 1;
      if (fit < a.B) a.slots = fit;
    }
  }
  if (a.slots > a.B) a.slots = a.B;
  if (a.state_only && (blocks || suffix || !a.Rout))
    return "state-only walk: needs a final-state buffer, no block states and no suffixes";
  // (with two visits per chunk only the first half of the state is handed over between sequences)
  if (a.slots < a.B && (!narrow || blocks || suffix))
    return "several batch entries per workgroup: only for the plain and state-only walks with dA of 64 or 128";
  return nullptr;
}

// Consecutive workgroup numbers go to the 8 XCDs in turn, and each XCD has an L2 of its own.  The
// workgroups that read the same rows should meet in one L2: the column tiles of a stream and, in a
// launch that holds several passes over the same tensors, the passes of a stream.  Launch index
// `block` of `passes * nwg` -> which pass (0 .. passes - 1) and which of its nwg workgroups.
struct WorkgroupId {
  int pass, wg;
};
FP_DEVICE WorkgroupId place_workgroup(int block, int nwg, int passes) {
  // XCD x runs the launch indices x, x + 8, ...; give it a contiguous range of the passes * nwg
  // logical numbers (one more for the first `rem` XCDs when 8 does not divide the total), in
  // which the passes of a workgroup and then the column tiles of a stream are neighbours.
  const int total = nwg * passes, per = total >> 3, rem = total & 7;
  const int xcd = block & 7, j = block >> 3;
  const int logical = xcd * per + (xcd < rem ? xcd : rem) + j;
  return WorkgroupId{logical % passes, logical / passes};
}

// Passes can share a launch if they walk the same shape in the same way (then they are the same
// kernel instantiation with the same grid); their tensors, direction and scales may differ.
inline bool same_walk(const PassArgs& a, const PassArgs& b) {
  return a.B == b.B && a.T == b.T && a.H == b.H && a.dA == b.dA && a.dB == b.dB && a.nblk == b.nblk &&
         a.block == b.block && a.Ls == b.Ls && a.state_only == b.state_only && a.slots == b.slots &&
         a.segs == b.segs && a.total == b.total &&
         (a.Bout != nullptr || a.Bin != nullptr) == (b.Bout != nullptr || b.Bin != nullptr) &&
         std::memcmp(a.log2g, b.log2g, sizeof a.log2g) == 0;
}

// Plans every pass of a launch and checks that they fit together.  Returns nullptr or a message.
inline const char* plan_passes(PassArgs* planned, const PassArgs* const* passes, int n, int compute_units) {
  if (n < 1 || n > MAX_PASSES_PER_LAUNCH) return "a launch holds one to three passes";
  for (int i = 0; i < n; ++i) {
    planned[i] = *passes[i];
    if (const char* why = plan_pass(planned[i], compute_units)) return why;
    if (i > 0 && !same_walk(planned[0], planned[i])) return "passes that share a launch must walk the same shape the same way";
  }
  return nullptr;
}

// Workgroups of a planned pass: a column tile of `slots` sequences each, or in the kernel of retention_pass_wide.h twice the columns of
// one sequence.
inline int pass_workgroups(const PassArgs& a) { return a.slots * a.H * (a.dB / BV); }
inline int wide_workgroups(const PassArgs& a) { return a.B * a.H * (a.dB / PW_D); }

// Whether everything that the kernels of retention_pass_fill.h and retention_pass_wide.h copy straight into LDS, 16 bytes at a time,
// starts at a multiple of them (rows and matrices are).  The pass kernel's loads into registers take any address.
inline bool copies_aligned(const PassArgs& a) {
  uintptr_t at = 0;
  for (const uint16_t* t : {a.X, a.W, a.Z, a.R0, a.R0lo, a.Bin, a.Xs, a.Ws, a.Zs}) at |= reinterpret_cast<uintptr_t>(t);
  return at % 16 == 0;
}

// Whether a pass of 64-wide keys over several sequences per workgroup, each of at most one chunk, takes the pass kernel's walk, whose rows go
// through registers: with one step a sequence, a step here (rows, a state in, a state out) is longer than there.  Speed of that walk over
// the kernel of retention_pass_fill.h, 256 units, by workgroups of 64 columns (sequences x heads x column tiles); inputs not in a cache /
// written by the launches right before:
//                     288            512            768            1024           1536           2048           4096
//   64 x 64   T40     1.06 / .95     1.06 / .97    1.06 / 1.20     1.05 / 1.16    1.01 / 1.08    .98            .92
//             T64     1.08 / 1.00    1.10 / 1.05   1.11 / 1.22     1.07 / 1.16    1.01 / 1.06    .98            .95
//   64 x 128  T64     1.07 / 1.01    1.05 / 1.09   1.03 / 1.18     1.01 / 1.18    .96 / 1.05     .95            .88
//   64 x 256  T64     1.05 / 1.01    1.06 / 1.01   1.04 / 1.15     1.02 / 1.12    .99 / 1.07     .93            .87
// Two chunks: .99 to 1.03 / 1.04 to 1.07 (64 x 64, 384 and 512), less beyond and with wider values.  Several passes in a launch (the backward's): .93
// to .98.
inline bool pass_is_short(const PassArgs& a, int passes, int compute_units) {
  return passes == 1 && a.T <= CH && (long long)a.B * a.H * (a.dB / BV) <= 6LL * compute_units;
}

// Calls run.template go<DA, MODE, NH>(slot), run.template fill<MODE>(slot) for the kernel of retention_pass_fill.h or run.wide(slot) for
// that of retention_pass_wide.h, for the instantiation that a launch of the `n` planned passes needs; `slot` numbers the
// instantiations 0 .. PASS_KERNELS - 1.
template <typename Run>
int dispatch_pass(const PassArgs* planned, int n, int compute_units, Run&& run) {
  const PassArgs& a = planned[0];
  bool copies = true;
  for (int i = 0; i < n; ++i) copies = copies && copies_aligned(planned[i]);
  const bool blocks = a.block > 0 && (a.Bout || a.Bin);
  const bool suffix = a.Ls > 0, multi = a.slots < a.B;
  // trailing tokens after the last block boundary, or suffixes in several parts: the general suffix walk
  const bool suffix_any = suffix && (a.T != a.nblk * a.block || a.Ls > CH);
  if (a.dA == 64) {
    if (copies && pop_folds(a)) return run.template fill<FILL_FOLD>(22);
    if (suffix_any) return run.template go<64, WALK_SUFFIX_ANY, 1>(14);
    if (suffix) return run.template go<64, WALK_SUFFIX, 1>(0);
    if (a.state_only) return run.template go<64, WALK_STATE, 1>(2);
    if (!copies) {
      if (blocks) return run.template go<64, WALK_BLOCKS, 1>(24);
      if (multi) return run.template go<64, WALK_MULTI, 1>(25);
      return run.template go<64, WALK_PLAIN, 1>(26);
    }
    if (blocks) return run.template fill<FILL_BLOCKS>(1);
    if (multi && pass_is_short(a, n, compute_units)) return run.template go<64, WALK_MULTI, 1>(25);
    if (multi) return run.template fill<FILL_MULTI>(3);
    return run.template fill<FILL_PLAIN>(4);
  }
  if (a.dA == 128) {
    if (suffix_any) return run.template go<128, WALK_SUFFIX_ANY, 1>(15);
    if (suffix) return run.template go<128, WALK_SUFFIX, 1>(5);
    if (blocks) return run.template go<128, WALK_BLOCKS, 1>(6);
    if (a.state_only) return run.template go<128, WALK_STATE, 1>(7);
    if (copies && pass_is_wide(a, n, compute_units)) return run.wide(23);
    if (multi) return run.template go<128, WALK_MULTI, 1>(8);
    return run.template go<128, WALK_PLAIN, 1>(9);
  }
  if (a.dA == 192) {   // three visits per chunk, 64 of the 192 contraction columns each
    if (suffix_any) return run.template go<64, WALK_SUFFIX_ANY, 3>(17);
    if (suffix) return run.template go<64, WALK_SUFFIX, 3>(18);
    if (a.state_only) return run.template go<64, WALK_STATE, 3>(19);
    if (blocks) return run.template go<64, WALK_BLOCKS, 3>(20);
    return run.template go<64, WALK_PLAIN, 3>(21);
  }
  // dA = 256: two visits per chunk, 128 of the 256 contraction columns each
  if (suffix_any) return run.template go<128, WALK_SUFFIX_ANY, 2>(16);
  if (suffix) return run.template go<128, WALK_SUFFIX, 2>(12);
  if (a.state_only) return run.template go<128, WALK_STATE, 2>(13);
  if (blocks) return run.template go<128, WALK_BLOCKS, 2>(10);
  return run.template go<128, WALK_PLAIN, 2>(11);
}

}  // namespace fpk
