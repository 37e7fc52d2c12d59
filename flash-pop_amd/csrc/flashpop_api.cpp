// C-ABI layer: argument checks and the mapping of retention forward / backward onto
// launches of the one pass kernel.  No device code and no HIP calls here.
//
// With s = dk^-1/2, A = s (q k^T) . D and P = s (dO v^T) . D (D the causal decay mask):
//
//   pass   X    W    Z    Y    R (dA x dB)        walk      s_intra s_read s_update
//   fwd    q    k    v    o    S      dk x dv     forward   s       1      s
//   dq     dO   v    k    dq   S^T    dv x dk     forward   s       1      s
//   dk     v    dO   q    dk   dS^T   dv x dk     backward  s       s      1
//   dv     k    q    dO   dv   dS     dk x dv     backward  s       s      1
//
// The column dimension dB is split over workgroups, the contraction dimension dA never is,
// so no pass needs a cross-workgroup reduction.  The dq pass re-runs the state recurrence
// instead of reading stored chunk states; the dk and dv passes each carry dS.  The three gradient
// passes are independent of each other and share launches where they fit (run_gradients).
//
// The POP entry points add block states to these passes (written by fwd, their gradients read
// by dk and dv); the fused POP entry points add the suffix tensors in the same four roles; the
// split entry points run the passes on segments of the sequences after a state-only pass and a
// scan; the decode step and the two elementwise stages around the op (rotary embedding of q and
// k, per-head normalisation with the swish gate) are kernels of their own.
#include "../../include/flashpop_hip.h"

#include <atomic>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <cstdint>
#include <cstdlib>
#include <mutex>

#include "pass_args.h"

namespace {

thread_local char g_err[256] = "";

int fail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof g_err, fmt, ap);
  va_end(ap);
  return code;
}

bool dim_ok(int d) { return d == 64 || d == 128 || d == 192 || d == 256; }

// Two measurement switches, read from the environment once per process (the first entry point that
// looks) and changed afterwards only through fp_set_backward_choice:
//   FLASHPOP_BWD   auto | passes | fused | paced   which backward runs where both exist (paced: fused, its two
//                  workgroups per stream held together, see FusedBwdArgs::want_pace)
//   FLASHPOP_CKPT  tokens between the checkpoints that the forward leaves for the fused backward
//                  (a multiple of 64; 0: none; unset: 512)
// A value that is neither is an error of every entry point, not a silent default.
enum BwdChoice { BWD_AUTO = 0, BWD_PASSES = 1, BWD_FUSED = 2, BWD_FUSED_PACED = 3 };
constexpr int kDefaultCheckpointEvery = 8 * fpk::CH;
std::atomic<int> g_bwd_choice{BWD_AUTO}, g_ckpt_every{kDefaultCheckpointEvery};
std::once_flag g_env_once;
char g_env_error[160] = "";

void read_environment() {
  std::call_once(g_env_once, [] {
    if (const char* e = std::getenv("FLASHPOP_BWD")) {
      if (std::strcmp(e, "passes") == 0) g_bwd_choice = BWD_PASSES;
      else if (std::strcmp(e, "fused") == 0) g_bwd_choice = BWD_FUSED;
      else if (std::strcmp(e, "paced") == 0) g_bwd_choice = BWD_FUSED_PACED;
      else if (std::strcmp(e, "auto") != 0 && *e)
        std::snprintf(g_env_error, sizeof g_env_error, "FLASHPOP_BWD=%.40s: expected auto, passes, fused or paced", e);
    }
    if (const char* e = std::getenv("FLASHPOP_CKPT")) {
      char* end = nullptr;
      const long n = std::strtol(e, &end, 10);
      if (end == e || *end || n < 0 || n % fpk::CH != 0 || n > (1 << 24))
        std::snprintf(g_env_error, sizeof g_env_error, "FLASHPOP_CKPT=%.40s: expected a non-negative multiple of %d", e, fpk::CH);
      else g_ckpt_every = (int)n;
    }
  });
}

struct Shape {
  int B, T, H, dk, dv;
  int segs = 0, total = 0;   // the B sequences are segments that do not divide theirs evenly (PassArgs)
};

int check_shape(const Shape& s, const double* decays) {
  read_environment();
  if (g_env_error[0]) return fail(FP_ERR_BAD_CONFIG, "%s", g_env_error);
  if (!decays) return fail(FP_ERR_NULL_POINTER, "head_decays is NULL");
  if (s.B < 1 || s.T < 1 || s.H < 1) return fail(FP_ERR_BAD_SHAPE, "B, T, H must be >= 1 (got %d, %d, %d)", s.B, s.T, s.H);
  if (s.H > fpk::MAX_HEADS) return fail(FP_ERR_BAD_SHAPE, "H = %d exceeds the supported maximum %d", s.H, fpk::MAX_HEADS);
  if (!dim_ok(s.dk) || !dim_ok(s.dv))
    return fail(FP_ERR_UNSUPPORTED_DIM, "dk and dv must be 64, 128, 192 or 256 (got dk=%d, dv=%d)", s.dk, s.dv);
  // per-tensor element counts are indexed with size_t in the kernel; the grid is an int
  // the kernels address one (batch, head) stream with 32-bit byte offsets
  const long long span = 2LL * s.T * s.H * (s.dk > s.dv ? s.dk : s.dv);
  if (span >= (1LL << 32)) return fail(FP_ERR_BAD_SHAPE, "T * H * max(dk, dv) too large: one sequence must stay below 4 GiB");
  // ... and a row of a tensor by a 32-bit index
  if ((long long)s.B * s.T >= (1LL << 32)) return fail(FP_ERR_BAD_SHAPE, "B * T too large: a tensor must have fewer than 2^32 rows");
  const long long wgs = (long long)s.B * s.H * ((s.dk > s.dv ? s.dk : s.dv) / fpk::BV);
  if (wgs > 0x7fffffffLL) return fail(FP_ERR_BAD_SHAPE, "B * H too large");
  for (int h = 0; h < s.H; ++h) {
    if (!(decays[h] > 0.0) || !(decays[h] <= 1.0))
      return fail(FP_ERR_BAD_DECAY, "head_decays[%d] = %g is outside (0, 1]", h, decays[h]);
  }
  return FP_OK;
}

// The pass kernels must not be recorded into a HIP graph (instantiating a graph that holds them has
// crashed the host process); the entry points that launch them refuse a capturing stream.
int check_stream(void* stream, const char* what) {
  if (fpk_stream_is_capturing(stream))
    return fail(FP_ERR_LAUNCH, "%s: the stream is capturing a HIP graph; this entry point must be called eagerly", what);
  return FP_OK;
}

void fill_common(fpk::PassArgs& a, const Shape& s, const double* decays) {
  std::memset(&a, 0, sizeof a);
  a.B = s.B;
  a.T = s.T;
  a.H = s.H;
  a.segs = s.segs;
  a.total = s.total;
  // log2(gamma) from the double, so gammas that round to 1.0f keep their decay
  for (int h = 0; h < s.H; ++h) a.log2g[h] = (float)std::log2(decays[h]);
}

bool misaligned(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) != 0; }
const uint16_t* in(const void* p) { return static_cast<const uint16_t*>(p); }
uint16_t* out(void* p) { return static_cast<uint16_t*>(p); }

int run(const fpk::PassArgs& a, void* stream, const char* what) {
  const char* msg = "";
  if (fpk_launch_pass(a, stream, &msg) != 0) return fail(FP_ERR_LAUNCH, "%s pass: %s", what, msg);
  return FP_OK;
}

// Independent passes over the same shape may share a launch (fpk_launch_passes).
bool same_launch(const fpk::PassArgs& x, const fpk::PassArgs& y) {
  return x.dA == y.dA && x.dB == y.dB && x.block == y.block && x.nblk == y.nblk && x.Ls == y.Ls &&
         (x.Bin != nullptr || x.Bout != nullptr) == (y.Bin != nullptr || y.Bout != nullptr);
}

int run_together(const fpk::PassArgs* const* passes, int n, void* stream, const char* what) {
  const char* msg = "";
  if (fpk_launch_passes(passes, n, stream, &msg) != 0) return fail(FP_ERR_LAUNCH, "%s passes: %s", what, msg);
  return FP_OK;
}

// The three gradient passes do not depend on each other.  How they are grouped into launches:
//  - dk and dv read the same q and dO rows walking backward; with dk == dv they are the same
//    kernel with the same grid, and in one launch the workgroups of a stream in both passes run
//    side by side, so those rows come from HBM once;
//  - dq has the shape of the dk pass.  Where one pass alone leaves compute units idle it joins
//    that launch (it walks the other way, so nothing is shared but the chip);
//  - what does not fit together (different dk and dv; block states in dk and dv but not in dq)
//    is launched on its own.
int run_gradients(const fpk::PassArgs& dq, const fpk::PassArgs& dk, const fpk::PassArgs& dv, void* stream,
                  const char* what) {
  const long long alone = (long long)dk.B * dk.H * (dk.dB / fpk::BV);   // workgroups of one pass
  const bool fills = alone >= fpk_compute_units();
  const bool dq_dk = same_launch(dq, dk), dk_dv = same_launch(dk, dv);
  if (dq_dk && dk_dv && !fills) {
    const fpk::PassArgs* all[] = {&dk, &dv, &dq};
    return run_together(all, 3, stream, what);
  }
  if (dk_dv) {
    if (int rc = run(dq, stream, what)) return rc;
    const fpk::PassArgs* both[] = {&dk, &dv};
    return run_together(both, 2, stream, what);
  }
  if (dq_dk && !fills) {
    const fpk::PassArgs* both[] = {&dq, &dk};
    if (int rc = run_together(both, 2, stream, what)) return rc;
    return run(dv, stream, what);
  }
  if (int rc = run(dq, stream, what)) return rc;
  if (int rc = run(dk, stream, what)) return rc;
  return run(dv, stream, what);
}

// dk and dv alone (the split-sequence backward runs its dq earlier)
int run_dk_dv(const fpk::PassArgs& dk, const fpk::PassArgs& dv, void* stream, const char* what) {
  if (same_launch(dk, dv)) {
    const fpk::PassArgs* both[] = {&dk, &dv};
    return run_together(both, 2, stream, what);
  }
  if (int rc = run(dk, stream, what)) return rc;
  return run(dv, stream, what);
}

// R = S, dk x dv, rows contiguous in dv
void plain_state(fpk::PassArgs& a, const Shape& s) {
  a.dA = s.dk;
  a.dB = s.dv;
  a.rs_a = s.dv;
  a.rs_n = 1;
}
// R = S^T, dv x dk, read through the strides of S
void transposed_state(fpk::PassArgs& a, const Shape& s) {
  a.dA = s.dv;
  a.dB = s.dk;
  a.rs_a = 1;
  a.rs_n = s.dv;
}

// Sequences of at most fpk::SS_ROWS tokens with head dimensions of 64 or 128: the forward that takes a (sequence,
// head) pair per step (short_seq.h) instead of a 64-token item per pair and column tile.  Shares the switch of the
// backward (the pass kernel stays reachable for comparisons).
bool fused_dim(int d);
bool use_short_forward(const Shape& s) {
  if (s.T > fpk::SS_ROWS || !fused_dim(s.dk) || !fused_dim(s.dv)) return false;
  read_environment();
  return g_bwd_choice.load(std::memory_order_relaxed) != BWD_PASSES;
}

int forward_short(const Shape& s, const void* q, const void* k, const void* v, const void* s0, const double* decays, void* o,
                  void* s_out, void* stream) {
  fpk::ShortFwdArgs a;
  std::memset(&a, 0, sizeof a);
  a.q = in(q); a.k = in(k); a.v = in(v); a.s0 = in(s0);
  a.o = out(o); a.s_out = out(s_out);
  a.B = s.B; a.T = s.T; a.H = s.H;
  a.dk_dim = s.dk; a.dv_dim = s.dv;
  a.scale = 1.0f / std::sqrt((float)s.dk);
  for (int h = 0; h < s.H; ++h) a.log2g[h] = (float)std::log2(decays[h]);
  const char* msg = "";
  if (fpk_launch_short_fwd(a, stream, &msg) != 0) return fail(FP_ERR_LAUNCH, "short-sequence forward: %s", msg);
  return FP_OK;
}

int forward(const Shape& s, const void* q, const void* k, const void* v, const void* s0, const double* decays, void* o,
            void* s_out, void* block_states, int block, void* stream, const uint16_t* s0_lo = nullptr) {
  if (!block_states && block == 0 && !s0_lo && use_short_forward(s)) return forward_short(s, q, k, v, s0, decays, o, s_out, stream);
  fpk::PassArgs a;
  fill_common(a, s, decays);
  const float sc = 1.0f / std::sqrt((float)s.dk);
  a.X = in(q); a.W = in(k); a.Z = in(v); a.Y = out(o);
  a.R0 = in(s0); a.R0lo = s0_lo; a.Rout = out(s_out); a.Bout = out(block_states);
  plain_state(a, s);
  a.block = block;
  a.nblk = block > 0 ? s.T / block : 0;
  a.reverse = 0;
  a.s_intra = sc; a.s_read = 1.f; a.s_update = sc;
  return run(a, stream, "forward");
}

// The plain backward with dk and dv of 64 or 128 has a kernel of its own that reads q, k, v, dO once for dk
// and dv together (retention_bwd_fused.h); it runs two workgroups per (batch, head) stream, so it
// is chosen when there are enough streams for the device (below).  The backward choice (FLASHPOP_BWD,
// fp_set_backward_choice) overrides that (for A/B measurements).
bool fused_dim(int d) { return d == 64 || d == 128; }
// `d_blocks` with `block`: gradients of POP block states arrive; the kernel adds them on its way when the blocks are
// whole chunks.
bool use_fused_backward(const Shape& s, const void* d_blocks, bool pop_suffixes = false, int block = 0) {
  if (!fused_dim(s.dk) || !fused_dim(s.dv)) return false;
  if (d_blocks && (block <= 0 || block % fpk::CH != 0)) return false;
  read_environment();
  const int choice = g_bwd_choice.load(std::memory_order_relaxed);
  if (choice == BWD_PASSES) return false;
  if (choice >= BWD_FUSED) return true;   // whatever the length and the number of streams
  if (s.T < 8 * fpk::CH) return false;    // short sequences: the walk over many of them per workgroup serves better
  // Two workgroups per stream against column-tiled passes that fill the chip: the fused kernel needs enough streams.
  // Measured cross-overs on a 256-unit device (forward + backward at T = 2048 .. 4096; streams = B * H):
  //                 dk = dv = 128      dk 64, dv 128      dk 128, dv 64      dk = dv = 64
  //   plain         86  (3 s >= CU)    32  (8 s >= CU)    64  (4 s >= CU)    64  (4 s >= CU)
  //   POP suffixes  48  (16 s >= 3 CU) 32  (8 s >= CU)    32  (8 s >= CU)    96  (8 s >= 3 CU)
  // (d = 128, 64 streams: 0.33 ms fused against 0.30 ms in passes at T = 4096; with suffixes the passes pay for every
  // suffix as a stop of each of their four walks and this kernel does not: 48 streams, 64-token blocks, 0.44 against
  // 0.57 ms.  Narrower states make the fused kernel's chunk step cheaper sooner than they help the passes.)
  const long long streams = (long long)s.B * s.H, cu = fpk_compute_units();
  const bool wide = s.dk == fpk::FB_D && s.dv == fpk::FB_D, narrow = s.dk == 64 && s.dv == 64;
  if (pop_suffixes) return wide ? 16 * streams >= 3 * cu : narrow ? 8 * streams >= 3 * cu : 8 * streams >= cu;
  return wide ? 3 * streams >= cu : s.dk == 64 && s.dv == fpk::FB_D ? 8 * streams >= cu : 4 * streams >= cu;
}

// Tokens between the states that fp_retention_fwd_ckpt leaves for the backward (0: none wanted).
// Eight chunks: the checkpoints cost 1/16 of the forward's traffic, and the segment that the two
// workgroups of a stream share stays within reach of the caches.
int checkpoint_interval(const Shape& s) {
  read_environment();
  const int every = g_ckpt_every.load(std::memory_order_relaxed);
  if (every <= 0 || !use_fused_backward(s, nullptr) || s.T <= every) return 0;
  return every;
}

// Suffix tensors of one fused POP call, in the roles q, k, v / d_o (inputs) and o / dq, dk, dv (outputs)
struct Suffixes {
  const void *q, *k, *v;
  int len;
};
struct SuffixGrads {
  const void* d_o;
  void *dq, *dk, *dv;
  int block;
};

int backward_fused(const Shape& s, const void* q, const void* k, const void* v, const void* s0, const double* decays,
                   const void* d_o, const void* d_s_out, void* dq, void* dk_, void* dv_, void* d_s0, void* stream,
                   const void* ckpt = nullptr, int ckpt_every = 0, const Suffixes* sfx = nullptr,
                   const SuffixGrads* sg = nullptr, const void* d_blocks = nullptr, int blocks_every = 0) {
  fpk::FusedBwdArgs a;
  std::memset(&a, 0, sizeof a);
  a.d_blocks = in(d_blocks);
  a.blocks_every = d_blocks ? blocks_every : 0;
  a.ckpt = in(ckpt);
  a.ckpt_every = ckpt ? ckpt_every : 0;
  a.want_pace = g_bwd_choice.load(std::memory_order_relaxed) == BWD_FUSED_PACED;
  if (sfx) {
    a.q_sfx = in(sfx->q); a.k_sfx = in(sfx->k); a.v_sfx = in(sfx->v); a.dO_sfx = in(sg->d_o);
    a.dq_sfx = out(sg->dq); a.dk_sfx = out(sg->dk); a.dv_sfx = out(sg->dv);
    a.block = sg->block;
    a.Ls = sfx->len;
  }
  a.q = in(q); a.k = in(k); a.v = in(v); a.dO = in(d_o);
  a.dq = out(dq); a.dk = out(dk_); a.dv = out(dv_);
  a.s0 = in(s0); a.ds_out = in(d_s_out); a.ds0 = out(d_s0);
  a.B = s.B; a.T = s.T; a.H = s.H;
  a.dk_dim = s.dk; a.dv_dim = s.dv;
  a.scale = 1.0f / std::sqrt((float)s.dk);
  for (int h = 0; h < s.H; ++h) a.log2g[h] = (float)std::log2(decays[h]);
  const char* msg = "";
  if (fpk_launch_bwd_fused(a, stream, &msg) != 0) return fail(FP_ERR_LAUNCH, "fused backward: %s", msg);
  return FP_OK;
}

// Many short sequences that each read a state of their own and whose final states nobody differentiates (the
// suffix call of the reference's POP layer): one kernel that takes a (sequence, head) pair per step (short_seq.h)
// instead of a 64-token item per pass and pair.
bool use_short_backward(const Shape& s, const void* d_s_out, const void* d_blocks) {
  if (s.T > fpk::SS_ROWS || d_s_out || d_blocks || !fused_dim(s.dk) || !fused_dim(s.dv)) return false;
  read_environment();
  return g_bwd_choice.load(std::memory_order_relaxed) != BWD_PASSES;
}

int backward_short(const Shape& s, const void* q, const void* k, const void* v, const void* s0, const double* decays,
                   const void* d_o, void* dq, void* dk_, void* dv_, void* d_s0, void* stream) {
  fpk::FusedBwdArgs a;
  std::memset(&a, 0, sizeof a);
  a.q = in(q); a.k = in(k); a.v = in(v); a.dO = in(d_o);
  a.dq = out(dq); a.dk = out(dk_); a.dv = out(dv_);
  a.s0 = in(s0); a.ds0 = out(d_s0);
  a.B = s.B; a.T = s.T; a.H = s.H;
  a.dk_dim = s.dk; a.dv_dim = s.dv;
  a.scale = 1.0f / std::sqrt((float)s.dk);
  for (int h = 0; h < s.H; ++h) a.log2g[h] = (float)std::log2(decays[h]);
  const char* msg = "";
  if (fpk_launch_short_bwd(a, stream, &msg) != 0) return fail(FP_ERR_LAUNCH, "short-sequence backward: %s", msg);
  return FP_OK;
}

int backward(const Shape& s, const void* q, const void* k, const void* v, const void* s0, const double* decays,
             const void* d_o, const void* d_s_out, const void* d_blocks, int block, void* dq, void* dk_, void* dv_,
             void* d_s0, void* stream) {
  if (use_short_backward(s, d_s_out, d_blocks)) return backward_short(s, q, k, v, s0, decays, d_o, dq, dk_, dv_, d_s0, stream);
  if (use_fused_backward(s, d_blocks, false, block) && !(d_blocks && d_s_out))
    return backward_fused(s, q, k, v, s0, decays, d_o, d_s_out, dq, dk_, dv_, d_s0, stream, nullptr, 0, nullptr, nullptr,
                          d_blocks, block);
  const float sc = 1.0f / std::sqrt((float)s.dk);
  const int nblk = block > 0 ? s.T / block : 0;
  fpk::PassArgs g, a;

  fill_common(g, s, decays);   // dq
  g.X = in(d_o); g.W = in(v); g.Z = in(k); g.Y = out(dq);
  g.R0 = in(s0);
  transposed_state(g, s);
  g.reverse = 0;
  g.s_intra = sc; g.s_read = 1.f; g.s_update = sc;

  fill_common(a, s, decays);   // dk
  a.X = in(v); a.W = in(d_o); a.Z = in(q); a.Y = out(dk_);
  a.R0 = in(d_s_out); a.Bin = in(d_blocks);
  transposed_state(a, s);
  a.block = d_blocks ? block : 0; a.nblk = nblk;
  a.reverse = 1;
  a.s_intra = sc; a.s_read = sc; a.s_update = 1.f;

  fpk::PassArgs b;
  fill_common(b, s, decays);   // dv (+ d_s0)
  b.X = in(k); b.W = in(q); b.Z = in(d_o); b.Y = out(dv_);
  b.R0 = in(d_s_out); b.Bin = in(d_blocks); b.Rout = out(d_s0);
  plain_state(b, s);
  b.block = d_blocks ? block : 0; b.nblk = nblk;
  b.reverse = 1;
  b.s_intra = sc; b.s_read = sc; b.s_update = 1.f;
  return run_gradients(g, a, b, stream, "gradient");
}

// ---- long sequences, few streams: cut every sequence into segments ---------------------------
// One workgroup walks one (batch, head, column tile) stream from end to end, so B * H * tiles
// workgroups is all the parallelism a pass has.  When that leaves most of the chip idle, each
// sequence is cut into S segments of whole chunks that run as separate sequences (all equally long but the last, which
// takes what is left):
//   1. a state-only pass gives the state each segment contributes on its own,
//   2. a scan over the S contributions gives the state at the start of every segment,
//   3. the ordinary pass runs on B * S sequences from those states.
// The backward does the same for S (needed by the dq pass; the forward's, or recomputed) and, walking
// backward, for dS.  The states of equal segments pass through bf16 like POP block states do, those of uneven ones and of
// POP blocks stay fp32 (Workspace).

// Tokens per segment for at most `target` segments (or segments of kMinChunks, the shortest worth a workgroup).
constexpr int kMinChunks = 4;
int segment_tokens(const Shape& s, long long target) {
  const long long chunks = (s.T + fpk::CH - 1LL) / fpk::CH, each = (chunks + target - 1) / target;
  return (int)(each > kMinChunks ? each : kMinChunks) * fpk::CH;
}
int segment_count(const Shape& s, int tokens) { return (int)((s.T + tokens - 1LL) / tokens); }

long long waves(long long workgroups) { return (workgroups + fpk_compute_units() - 1) / fpk_compute_units(); }

// The segments that fill the chip once (1: do not cut), for a call that uncut would leave at least two thirds of the compute
// units idle in its narrowest pass.  Equally long ones are taken where there are some that are at most a quarter longer
// than the shortest possible (a chunk step or two against a longer scan and more segment states).
int plan_segments(const Shape& s) {
  const int tiles = (s.dk < s.dv ? s.dk : s.dv) / fpk::BV;
  const long long target = fpk_compute_units() / ((long long)s.B * s.H * tiles);
  if (target < 3) return 1;
  const int chunks = (int)((s.T + fpk::CH - 1LL) / fpk::CH), tokens = segment_tokens(s, target);
  int even = 1;
  for (int n = 2; n <= target && n <= chunks; ++n) {
    if (s.T % fpk::CH == 0 && chunks % n == 0 && chunks / n >= kMinChunks) even = n;
  }
  return even > 1 && 4 * (chunks / even) * fpk::CH <= 5 * tokens ? even : segment_count(s, tokens);
}
// Whether n segments shorten the chain of chunk steps by what the cut costs: its extra launches, and the segment states
// that it moves.  Forward on the 256-unit device, launches in a row, a step there 0.72 us (64-wide keys) or 1.4 (128), uncut -> cut, *: the
// line cuts it:
//   64 x 64    H4 B1     13 chunks 12.9 -> 16.2 us   16 chunks 15.3 -> 15.2   18 chunks 16.6 -> 16.5*  28 chunks 23.8 -> 15.4*
//   64 x 64    H12 B6    28 chunks 24.6 -> 27.6      40 chunks 33.3 -> 33.6*  79 chunks 61.9 -> 53.6*
//   64 x 128   H12 B1    13 chunks 13.2 -> 17.7      18 chunks 17.0 -> 18.1   28 chunks 24.2 -> 17.3*  79 chunks 61.8 -> 29.2*
//   128 x 128  H8 B3     13 chunks 22.3 -> 25.5      18 chunks 29.1 -> 26.5   28 chunks 43.0 -> 29.1*
//   128 x 256  H8 B2     13 chunks 22.3 -> 27.4      18 chunks 29.2 -> 27.9   28 chunks 43.0 -> 26.9   40 chunks 59.8 -> 31.4*
// Backward (the uncut passes share launches, or are the fused kernel with its longer step; the cut has four launches and the
// forward's states):
//   64 x 64    H4 B1     18 chunks 16.6 -> 24.2      28 chunks 23.8 -> 22.5*  40 chunks 32.5 -> 22.8*
//   64 x 64    H12 B6    28 chunks 50.2 -> 51.2      40 chunks 69.7 -> 64.5*  79 chunks 133 -> 106* (uncut: fused)
//   64 x 128   H12 B1    13 chunks 35.0 -> 37.8      18 chunks 45.8 -> 38.4   28 chunks 67.6 -> 36.2*  79 chunks 178 -> 54.2*
//   128 x 128  H16 B1    18 chunks 29.3 -> 36.6      28 chunks 43.2 -> 35.3   40 chunks 60.2 -> 41.0*  79 chunks 116 -> 65.2*
//   128 x 256  H8 B2     13 chunks 58.5 -> 57.0      18 chunks 78.0 -> 59.0   28 chunks 117 -> 58.9    40 chunks 165 -> 70.2*
// The line is that of slower kernels on both sides.  Of these rows none that it cuts is slower for it by more than 1 %; what it leaves uncut would be
// shorter cut from 18 chunks of 128-wide keys on in the forward (128 x 256, 28 chunks: by 16 us), from 28 (128 x 128), 18 (64 x 128) and 18
// (128 x 256: by up to 58 us) in the backward.
// `block`: a POP call, whose chunks end at its blocks and whose gradient passes share fewer launches (64 x 128, B4 H4 T1440
// in blocks of 144, 30 chunks, with the suffix call and the launches between the two: 200 -> 166 us).
bool cut_pays(const Shape& s, int n, int tokens, bool backward, int block = 0) {
  const int launch = fpk_launch_steps();   // what a launch costs, in chunk steps
  if (launch <= 0) return true;
  const long long each = (tokens + fpk::CH - 1) / fpk::CH, chunks = block > 0 ? n * each : (s.T + fpk::CH - 1LL) / fpk::CH;
  const long long streams = (long long)s.B * s.H * n, tk = s.dk / fpk::BV, tv = s.dv / fpk::BV;
  const double matrix = s.dk * s.dv / 16384.;
  const long long contrib = waves(streams * (s.dk == fpk::FB_D && s.dv % fpk::FB_D == 0 ? s.dv / fpk::FB_D : tv));
  if (!backward) return chunks - each * (contrib + waves(streams * tv)) >= launch * (2 + 1.25 * matrix);
  const long long dk_dv = s.dk == s.dv ? waves(2 * streams * tk) : waves(streams * tk) + waves(streams * tv);
  const bool fused = use_fused_backward(s, nullptr) && block % fpk::CH == 0;
  const long long uncut = fused ? 7 * chunks / 4 : ((s.dk == s.dv ? 1 : 2) + (block > 0 ? 1 : 0)) * chunks;
  return uncut - each * (contrib + waves(streams * tk) + dk_dv) >= launch * (2.5 + 1.75 * matrix);
}
// Forward and backward cut a sequence the same way, so that the states the forward leaves at the start of every segment
// are the ones the backward's dq pass needs; a backward is cut only if its forward is.
int plan_forward(const Shape& s) {
  const int n = plan_segments(s);
  return n > 1 && cut_pays(s, n, segment_tokens(s, n), false) ? n : 1;
}
int plan_backward(const Shape& s) {
  const int n = plan_forward(s);
  return n > 1 && cut_pays(s, n, segment_tokens(s, n), true) ? n : 1;
}

// Whether the bytes that a POP call cut at its blocks moves are worth the chain they replace: q, k, v, o, k and v a second time,
// and per element of a block's state 18 bytes (fp32 written, read and written by the scan, read; bf16 out), where the uncut call
// moves 2.  There are as many states as blocks, however many fill the chip, and the cut call streams them at 3.5 to 4.8 TB/s
// while the uncut one walks, 1.2 to 1.3 us a chunk with 64-wide keys, 1.9 to 2.2 with 128: 6.8 MB a step tell the two apart (three steps:
// the launches).  Uncut -> cut, forward / backward, us, launches in a row, *: the line cuts it:
//   128 x 128  blocks of 64    B10 H4 T4096   130 -> 211 / 227 -> 332      B4 H4 T4096   130 -> 115* / 226 -> 154*
//   128 x 128  blocks of 144   B10 H4 T16384  597 -> 559 / 933 -> 973      B4 H8 T4096   146 -> 117* / 238 -> 205*
//   64 x 128   blocks of 64    B6 H8 T4096     80 -> 126 / 192 -> 245      B6 H4 T2048    42 -> 49* / 155 -> 83*
//   64 x 64    blocks of 64    B10 H8 T4096    80 -> 116 / 158 -> 222      B6 H8 T16384  334 -> 382* / 541 -> 578*
// The line is from when a chunk of 64-wide keys took 1.5 to 1.7 us: it now cuts some of those calls that walk as fast or faster (the
// last two rows' right).
bool block_states_pay(const Shape& s, int segments, int block) {
  if (fpk_launch_steps() <= 0) return true;   // (a device whose launches cost nothing)
  const double chunks = (double)segments * ((block + fpk::CH - 1) / fpk::CH);
  const double bytes = 6.0 * s.B * s.T * s.H * (s.dk + s.dv) + 18.0 * s.B * segments * s.H * s.dk * s.dv;
  return bytes <= 6.8e6 * (chunks - 3);
}

// Segments per sequence of a POP call (1: not cut), one per block and one for the tokens after the last block: the scan over
// the contributions then passes every block state, and the gradients of block states join in it, so that the passes are
// those of a plain call.  For the streams that a plain call is cut for, and blocks of at least a chunk (a shorter block
// has more state than tokens to move), where the chain gets shorter by what the cut costs and its states do not take longer to move.
int plan_pop_forward(const Shape& s, int block) {
  const long long streams = (long long)s.B * s.H * ((s.dk < s.dv ? s.dk : s.dv) / fpk::BV);
  if (block < fpk::CH || s.T <= block || 3 * streams > fpk_compute_units()) return 1;
  const int n = segment_count(s, block);
  return block_states_pay(s, n, block) && cut_pays(s, n, block, false, block) ? n : 1;
}
int plan_pop_backward(const Shape& s, int block) {
  const int n = plan_pop_forward(s, block);
  return n > 1 && cut_pays(s, n, block, true, block) ? n : 1;
}

size_t workspace_bytes(const Shape& s, int segments) {
  return segments > 1 ? 2 * sizeof(uint16_t) * (size_t)s.B * segments * s.H * s.dk * s.dv : 0;
}

struct Workspace {
  uint16_t* contrib;      // [B, S, H, dk, dv]: what each segment adds on its own
  uint16_t* start;        // [B, S, H, dk, dv]: state at the segment's first token (last, walking backward)
  // The lower halves of the two where they are fp32 (PassArgs::R0lo), nullptr: they are bf16.  With them the scan works in
  // place, so the bytes are the same either way.  Equal segments keep bf16 states (at B2 H8 T16384 128 x 256 fp32 ones would
  // be 5 % more traffic); where a sequence is cut unevenly or at its blocks the states stay fp32, as one walk carries them.
  uint16_t *contrib_lo, *start_lo;
};

Workspace carve(void* workspace, const Shape& s, const Shape& seg) {
  uint16_t* const base = static_cast<uint16_t*>(workspace);
  uint16_t* const second = base + (size_t)seg.B * s.H * s.dk * s.dv;
  return seg.segs > 0 ? Workspace{base, base, second, second} : Workspace{base, second, nullptr, nullptr};
}

// Block states of a POP call that is cut at its blocks: where the forward's scan leaves them, the gradients that the
// backward's scan meets
struct BlockStates {
  uint16_t* out;
  const uint16_t* in;
  int n;
};

int scan(const Shape& s, const Shape& seg, const double* decays, const Workspace& w, const void* r0, void* fin, int reverse,
         const BlockStates& blocks, void* stream) {
  fpk::ScanArgs a;
  std::memset(&a, 0, sizeof a);
  a.U = w.contrib; a.R0 = in(r0); a.init = w.start; a.fin = out(fin);
  a.U_lo = w.contrib_lo; a.init_lo = w.start_lo;
  a.blocks_out = blocks.out; a.blocks_in = blocks.in; a.nblk = blocks.n;
  a.B = s.B; a.S = seg.B / s.B; a.H = s.H; a.M = s.dk * s.dv; a.reverse = reverse;
  a.Tseg = seg.T;
  a.Tlast = s.T - (a.S - 1) * seg.T;
  for (int h = 0; h < s.H; ++h) a.log2g[h] = (float)std::log2(decays[h]);
  const char* msg = "";
  if (fpk_launch_scan(a, stream, &msg) != 0) return fail(FP_ERR_LAUNCH, "segment scan: %s", msg);
  return FP_OK;
}

// the B * S sequences that the segments form (the same memory, reinterpreted)
Shape segment_shape(const Shape& s, int segments) {
  const int tokens = segment_tokens(s, segments);
  const bool even = (long long)tokens * segments == s.T;
  return Shape{s.B * segments, tokens, s.H, s.dk, s.dv, even ? 0 : segments, even ? 0 : s.T};
}

// A POP call cut at its blocks: every block, and the tokens after the last one, a segment with fp32 states.
Shape block_segments(const Shape& s, int block) {
  const int segments = segment_count(s, block);
  return Shape{s.B * segments, block, s.H, s.dk, s.dv, segments, s.T};
}

// State-only pass: contributions of the segments to S (forward walk over k, v) or to dS
// (backward walk over q, dO).
int contributions(const Shape& seg, const double* decays, const void* w_rows, const void* z_rows, int reverse,
                  const Workspace& w, void* stream) {
  const float sc = 1.0f / std::sqrt((float)seg.dk);
  // the kernel that holds whole columns of the state per workgroup
  if (fpk::contrib_pays(seg.B, seg.T, seg.H, seg.dk, seg.dv, fpk_compute_units()) && fpk::contrib_fits(seg.T, seg.H, seg.dk, seg.dv)) {
    fpk::ContribArgs c;
    std::memset(&c, 0, sizeof c);
    c.W = in(w_rows); c.Z = in(z_rows); c.U = w.contrib; c.U_lo = w.contrib_lo;
    c.B = seg.B; c.T = seg.T; c.H = seg.H; c.dk = seg.dk; c.dB = seg.dv; c.reverse = reverse;
    c.segs = seg.segs; c.total = seg.total;
    c.s_update = reverse ? 1.f : sc;
    for (int h = 0; h < seg.H; ++h) c.log2g[h] = (float)std::log2(decays[h]);
    const char* msg = "";
    if (fpk_launch_contrib(c, stream, &msg) != 0) return fail(FP_ERR_LAUNCH, "%s: %s", reverse ? "dS contributions" : "S contributions", msg);
    return FP_OK;
  }
  fpk::PassArgs a;
  fill_common(a, seg, decays);
  a.X = in(w_rows);   // never read
  a.W = in(w_rows); a.Z = in(z_rows);
  a.Rout = w.contrib; a.Rout_lo = w.contrib_lo;
  plain_state(a, seg);
  a.reverse = reverse;
  a.state_only = 1;
  a.s_intra = sc; a.s_read = reverse ? sc : 1.f; a.s_update = reverse ? 1.f : sc;
  return run(a, stream, reverse ? "dS contributions" : "S contributions");
}

int forward_split(const Shape& s, const Shape& seg, const void* q, const void* k, const void* v, const void* s0,
                  const double* decays, void* o, void* s_out, void* workspace, void* stream, const BlockStates& blocks = {}) {
  const Workspace w = carve(workspace, s, seg);
  int rc;
  if ((rc = contributions(seg, decays, k, v, 0, w, stream)) != FP_OK) return rc;
  if ((rc = scan(s, seg, decays, w, s0, s_out, 0, blocks, stream)) != FP_OK) return rc;
  return forward(seg, q, k, v, w.start, decays, o, nullptr, nullptr, 0, stream, w.start_lo);
}

int backward_split(const Shape& s, const Shape& seg, const void* q, const void* k, const void* v, const void* s0,
                   const double* decays, const void* d_o, const void* d_s_out, void* dq, void* dk_, void* dv_,
                   void* d_s0, void* workspace, bool states_kept, void* stream, const BlockStates& blocks = {}) {
  const Workspace w = carve(workspace, s, seg);
  const float sc = 1.0f / std::sqrt((float)s.dk);
  fpk::PassArgs a;
  int rc;

  // S at the start of every segment (unless the forward's are still there), then dq
  if (!states_kept) {
    if ((rc = contributions(seg, decays, k, v, 0, w, stream)) != FP_OK) return rc;
    if ((rc = scan(s, seg, decays, w, s0, nullptr, 0, {}, stream)) != FP_OK) return rc;
  }
  fill_common(a, seg, decays);
  a.X = in(d_o); a.W = in(v); a.Z = in(k); a.Y = out(dq);
  a.R0 = w.start; a.R0lo = w.start_lo;
  transposed_state(a, seg);
  a.reverse = 0;
  a.s_intra = sc; a.s_read = 1.f; a.s_update = sc;
  if ((rc = run(a, stream, "dq")) != FP_OK) return rc;

  // dS at the end of every segment (the workspace is free again: the stream orders the passes), then dk and dv
  if ((rc = contributions(seg, decays, q, d_o, 1, w, stream)) != FP_OK) return rc;
  if ((rc = scan(s, seg, decays, w, d_s_out, d_s0, 1, blocks, stream)) != FP_OK) return rc;
  fill_common(a, seg, decays);
  a.X = in(v); a.W = in(d_o); a.Z = in(q); a.Y = out(dk_);
  a.R0 = w.start; a.R0lo = w.start_lo;
  transposed_state(a, seg);
  a.reverse = 1;
  a.s_intra = sc; a.s_read = sc; a.s_update = 1.f;

  fpk::PassArgs b;
  fill_common(b, seg, decays);
  b.X = in(k); b.W = in(q); b.Z = in(d_o); b.Y = out(dv_);
  b.R0 = w.start; b.R0lo = w.start_lo;
  plain_state(b, seg);
  b.reverse = 1;
  b.s_intra = sc; b.s_read = sc; b.s_update = 1.f;
  return run_dk_dv(a, b, stream, "dk / dv");
}

int check_workspace(const Shape& s, int segments, const void* workspace, size_t bytes, const char* query = "fp_retention_workspace_bytes") {
  if (segments <= 1) return FP_OK;
  if (!workspace) return fail(FP_ERR_NULL_POINTER, "workspace is NULL but %s() is nonzero for this shape", query);
  if (bytes < workspace_bytes(s, segments))
    return fail(FP_ERR_BAD_SHAPE, "workspace of %zu bytes is smaller than the %zu that %s() asks for", bytes,
                workspace_bytes(s, segments), query);
  if (reinterpret_cast<uintptr_t>(workspace) % 16 != 0) return fail(FP_ERR_BAD_SHAPE, "workspace must be 16-byte aligned");
  return FP_OK;
}

int check_fused(const Shape& s, int block, int sfx_len) {
  if (block < 1) return fail(FP_ERR_BAD_SHAPE, "block_size must be >= 1 (got %d)", block);
  if (sfx_len < 1) return fail(FP_ERR_BAD_SHAPE, "suffix length must be positive (got %d)", sfx_len);
  if (sfx_len > fpk::CH && (s.dk > 128 || s.dv > 128))
    return fail(FP_ERR_UNSUPPORTED_DIM, "suffixes longer than %d tokens need dk and dv of 64 or 128 (got %d, %d)", fpk::CH, s.dk, s.dv);
  if ((long long)s.B * (s.T / block + 1) * sfx_len >= (1LL << 32))
    return fail(FP_ERR_BAD_SHAPE, "too many suffix rows: B * (T / block_size + 1) * sfx_len must stay below 2^32");
  return FP_OK;
}

void suffix_walk(fpk::PassArgs& a, const Shape& s, int block, int sfx_len, const void* x, const void* w, const void* z,
                 void* y) {
  a.block = block;
  a.nblk = s.T / block;
  a.Ls = sfx_len;
  a.Xs = in(x); a.Ws = in(w); a.Zs = in(z); a.Ys = out(y);
}

int fused_forward(const Shape& s, const void* q, const void* k, const void* v, const void* s0, const Suffixes& x,
                  const double* decays, void* o, void* o_sfx, void* s_out, int block, void* stream) {
  fpk::PassArgs a;
  fill_common(a, s, decays);
  const float sc = 1.0f / std::sqrt((float)s.dk);
  a.X = in(q); a.W = in(k); a.Z = in(v); a.Y = out(o);
  a.R0 = in(s0); a.Rout = out(s_out);
  plain_state(a, s);
  suffix_walk(a, s, block, x.len, x.q, x.k, x.v, o_sfx);
  a.reverse = 0;
  a.s_intra = sc; a.s_read = 1.f; a.s_update = sc;
  return run(a, stream, "fused forward");
}

int fused_backward(const Shape& s, const void* q, const void* k, const void* v, const void* s0, const Suffixes& x,
                   const double* decays, const void* d_o, const void* d_o_sfx, const void* d_s_out, void* dq, void* dk_,
                   void* dv_, void* dq_sfx, void* dk_sfx, void* dv_sfx, void* d_s0, int block, void* stream) {
  // whole 64-token chunks per block, suffixes of one chunk at most: the kernel that carries dS once
  if (use_fused_backward(s, nullptr, true) && block % fpk::CH == 0 && s.T % block == 0 && x.len <= fpk::CH) {
    const SuffixGrads sg{d_o_sfx, dq_sfx, dk_sfx, dv_sfx, block};
    return backward_fused(s, q, k, v, s0, decays, d_o, d_s_out, dq, dk_, dv_, d_s0, stream, nullptr, 0, &x, &sg);
  }
  const float sc = 1.0f / std::sqrt((float)s.dk);
  fpk::PassArgs g, a;

  fill_common(g, s, decays);   // dq
  g.X = in(d_o); g.W = in(v); g.Z = in(k); g.Y = out(dq);
  g.R0 = in(s0);
  transposed_state(g, s);
  suffix_walk(g, s, block, x.len, d_o_sfx, x.v, x.k, dq_sfx);
  g.reverse = 0;
  g.s_intra = sc; g.s_read = 1.f; g.s_update = sc;

  fill_common(a, s, decays);   // dk
  a.X = in(v); a.W = in(d_o); a.Z = in(q); a.Y = out(dk_);
  a.R0 = in(d_s_out);
  transposed_state(a, s);
  suffix_walk(a, s, block, x.len, x.v, d_o_sfx, x.q, dk_sfx);
  a.reverse = 1;
  a.s_intra = sc; a.s_read = sc; a.s_update = 1.f;

  fpk::PassArgs b;
  fill_common(b, s, decays);   // dv (+ d_s0)
  b.X = in(k); b.W = in(q); b.Z = in(d_o); b.Y = out(dv_);
  b.R0 = in(d_s_out); b.Rout = out(d_s0);
  plain_state(b, s);
  suffix_walk(b, s, block, x.len, x.k, x.q, d_o_sfx, dv_sfx);
  b.reverse = 1;
  b.s_intra = sc; b.s_read = sc; b.s_update = 1.f;
  return run_gradients(g, a, b, stream, "fused gradient");
}

}  // namespace

extern "C" {

int fp_retention_fwd(const void* q, const void* k, const void* v, const void* s0, const double* head_decays, void* o,
                     void* s_out, int B, int T, int H, int dk, int dv, void* stream) {
  const Shape s{B, T, H, dk, dv};
  if (int rc = check_shape(s, head_decays)) return rc;
  if (int rc = check_stream(stream, "fp_retention_fwd")) return rc;
  if (!q || !k || !v || !o) return fail(FP_ERR_NULL_POINTER, "q, k, v and o must not be NULL");
  return forward(s, q, k, v, s0, head_decays, o, s_out, nullptr, 0, stream);
}

int fp_retention_bwd(const void* q, const void* k, const void* v, const void* s0, const double* head_decays,
                     const void* d_o, const void* d_s_out, void* dq, void* dk_, void* dv_, void* d_s0, int B, int T,
                     int H, int dk, int dv, void* stream) {
  const Shape s{B, T, H, dk, dv};
  if (int rc = check_shape(s, head_decays)) return rc;
  if (int rc = check_stream(stream, "fp_retention_bwd")) return rc;
  if (!q || !k || !v || !d_o || !dq || !dk_ || !dv_)
    return fail(FP_ERR_NULL_POINTER, "q, k, v, d_o, dq, dk and dv must not be NULL");
  return backward(s, q, k, v, s0, head_decays, d_o, d_s_out, nullptr, 0, dq, dk_, dv_, d_s0, stream);
}

size_t fp_retention_checkpoint_bytes(int B, int T, int H, int dk, int dv, int* every) {
  const Shape s{B, T, H, dk, dv};
  if (every) *every = 0;
  if (B < 1 || T < 1 || H < 1 || H > fpk::MAX_HEADS || !dim_ok(dk) || !dim_ok(dv)) return 0;
  const int n = checkpoint_interval(s);
  if (n <= 0) return 0;
  if (every) *every = n;
  return sizeof(uint16_t) * (size_t)B * (T / n) * H * dk * dv;
}

int fp_retention_fwd_ckpt(const void* q, const void* k, const void* v, const void* s0, const double* head_decays, void* o,
                          void* s_out, void* checkpoints, int every, int B, int T, int H, int dk, int dv, void* stream) {
  const Shape s{B, T, H, dk, dv};
  if (int rc = check_shape(s, head_decays)) return rc;
  if (int rc = check_stream(stream, "fp_retention_fwd_ckpt")) return rc;
  if (!q || !k || !v || !o) return fail(FP_ERR_NULL_POINTER, "q, k, v and o must not be NULL");
  if (!checkpoints || every <= 0) return forward(s, q, k, v, s0, head_decays, o, s_out, nullptr, 0, stream);
  if (every % fpk::CH != 0) return fail(FP_ERR_BAD_SHAPE, "the checkpoint interval must be a multiple of %d tokens (got %d)", fpk::CH, every);
  return forward(s, q, k, v, s0, head_decays, o, s_out, T / every > 0 ? checkpoints : nullptr, every, stream);
}

int fp_retention_bwd_ckpt(const void* q, const void* k, const void* v, const void* s0, const double* head_decays,
                          const void* d_o, const void* d_s_out, const void* checkpoints, int every, void* dq, void* dk_,
                          void* dv_, void* d_s0, int B, int T, int H, int dk, int dv, void* stream) {
  const Shape s{B, T, H, dk, dv};
  if (int rc = check_shape(s, head_decays)) return rc;
  if (int rc = check_stream(stream, "fp_retention_bwd_ckpt")) return rc;
  if (!q || !k || !v || !d_o || !dq || !dk_ || !dv_)
    return fail(FP_ERR_NULL_POINTER, "q, k, v, d_o, dq, dk and dv must not be NULL");
  if (checkpoints && (every <= 0 || every % fpk::CH != 0))
    return fail(FP_ERR_BAD_SHAPE, "the checkpoint interval must be a positive multiple of %d tokens (got %d)", fpk::CH, every);
  if (checkpoints && T / every > 0 && use_fused_backward(s, nullptr))
    return backward_fused(s, q, k, v, s0, head_decays, d_o, d_s_out, dq, dk_, dv_, d_s0, stream, checkpoints, every);
  return backward(s, q, k, v, s0, head_decays, d_o, d_s_out, nullptr, 0, dq, dk_, dv_, d_s0, stream);
}

size_t fp_retention_workspace_bytes(int B, int T, int H, int dk, int dv) {
  const Shape s{B, T, H, dk, dv};
  if (B < 1 || T < 1 || H < 1 || H > fpk::MAX_HEADS || !dim_ok(dk) || !dim_ok(dv)) return 0;
  return workspace_bytes(s, plan_forward(s));   // (a backward is cut as its forward, or not at all)
}

size_t fp_retention_backward_workspace_bytes(int B, int T, int H, int dk, int dv) {
  return fp_retention_workspace_bytes(B, T, H, dk, dv) ? workspace_bytes(Shape{B, T, H, dk, dv}, plan_backward(Shape{B, T, H, dk, dv})) : 0;
}

int fp_retention_fwd_split(const void* q, const void* k, const void* v, const void* s0, const double* head_decays,
                           void* o, void* s_out, int B, int T, int H, int dk, int dv, void* workspace,
                           size_t workspace_bytes_given, void* stream) {
  const Shape s{B, T, H, dk, dv};
  if (int rc = check_shape(s, head_decays)) return rc;
  if (int rc = check_stream(stream, "fp_retention_fwd_split")) return rc;
  if (!q || !k || !v || !o) return fail(FP_ERR_NULL_POINTER, "q, k, v and o must not be NULL");
  const int segments = plan_forward(s);
  if (int rc = check_workspace(s, segments, workspace, workspace_bytes_given)) return rc;
  if (segments <= 1) return forward(s, q, k, v, s0, head_decays, o, s_out, nullptr, 0, stream);
  return forward_split(s, segment_shape(s, segments), q, k, v, s0, head_decays, o, s_out, workspace, stream);
}

int fp_retention_fwd_split_static(const void* q, const void* k, const void* v, const void* s0,
                                  const double* head_decays, void* o, void* s_out, int B, int T, int H, int dk, int dv,
                                  void* stream) {
  const Shape s{B, T, H, dk, dv};
  if (int rc = check_shape(s, head_decays)) return rc;
  if (int rc = check_stream(stream, "fp_retention_fwd_split_static")) return rc;
  if (!q || !k || !v || !o) return fail(FP_ERR_NULL_POINTER, "q, k, v and o must not be NULL");
  const int segments = plan_forward(s);
  if (segments <= 1) return forward(s, q, k, v, s0, head_decays, o, s_out, nullptr, 0, stream);
  const size_t need = workspace_bytes(s, segments);
  if (need > fpk::STATIC_SCRATCH_BYTES)
    return fail(FP_ERR_BAD_SHAPE,
                "this shape needs %zu bytes of segment states, more than the %zu bytes of the library's own scratch: "
                "use fp_retention_fwd_split with a workspace",
                need, (size_t)fpk::STATIC_SCRATCH_BYTES);
  void* scratch_ptr = nullptr;
  const char* msg = "";
  if (fpk_static_scratch(&scratch_ptr, &msg) != 0) return fail(FP_ERR_LAUNCH, "%s", msg);
  // nothing in the scratch has to start at zero: the state-only pass writes every segment's
  // contribution and the scan every starting state before anything reads them
  return forward_split(s, segment_shape(s, segments), q, k, v, s0, head_decays, o, s_out, scratch_ptr, stream);
}

int fp_retention_bwd_split(const void* q, const void* k, const void* v, const void* s0, const double* head_decays,
                           const void* d_o, const void* d_s_out, void* dq, void* dk_, void* dv_, void* d_s0, int B,
                           int T, int H, int dk, int dv, void* workspace, size_t workspace_bytes_given,
                           int forward_states_kept, void* stream) {
  const Shape s{B, T, H, dk, dv};
  if (int rc = check_shape(s, head_decays)) return rc;
  if (int rc = check_stream(stream, "fp_retention_bwd_split")) return rc;
  if (!q || !k || !v || !d_o || !dq || !dk_ || !dv_)
    return fail(FP_ERR_NULL_POINTER, "q, k, v, d_o, dq, dk and dv must not be NULL");
  const int segments = plan_backward(s);
  if (int rc = check_workspace(s, segments, workspace, workspace_bytes_given)) return rc;
  if (segments <= 1) return backward(s, q, k, v, s0, head_decays, d_o, d_s_out, nullptr, 0, dq, dk_, dv_, d_s0, stream);
  return backward_split(s, segment_shape(s, segments), q, k, v, s0, head_decays, d_o, d_s_out, dq, dk_, dv_, d_s0, workspace,
                        forward_states_kept != 0, stream);
}

int fp_pop_retention_fwd(const void* q, const void* k, const void* v, const void* s0, const double* head_decays,
                         void* o, void* block_states, int B, int T, int H, int dk, int dv, int block_size,
                         void* stream) {
  const Shape s{B, T, H, dk, dv};
  if (int rc = check_shape(s, head_decays)) return rc;
  if (int rc = check_stream(stream, "fp_pop_retention_fwd")) return rc;
  if (block_size < 1) return fail(FP_ERR_BAD_SHAPE, "block_size must be >= 1 (got %d)", block_size);
  if (!q || !k || !v || !o) return fail(FP_ERR_NULL_POINTER, "q, k, v and o must not be NULL");
  if (!block_states && T / block_size > 0)
    return fail(FP_ERR_NULL_POINTER, "block_states is NULL but T / block_size = %d", T / block_size);
  return forward(s, q, k, v, s0, head_decays, o, nullptr, block_states, block_size, stream);
}

size_t fp_pop_retention_workspace_bytes(int B, int T, int H, int dk, int dv, int block_size) {
  const Shape s{B, T, H, dk, dv};
  if (B < 1 || T < 1 || H < 1 || H > fpk::MAX_HEADS || !dim_ok(dk) || !dim_ok(dv) || block_size < 1) return 0;
  return workspace_bytes(s, plan_pop_forward(s, block_size));
}

size_t fp_pop_retention_backward_workspace_bytes(int B, int T, int H, int dk, int dv, int block_size) {
  const Shape s{B, T, H, dk, dv};
  return fp_pop_retention_workspace_bytes(B, T, H, dk, dv, block_size) ? workspace_bytes(s, plan_pop_backward(s, block_size)) : 0;
}

int fp_pop_retention_fwd_split(const void* q, const void* k, const void* v, const void* s0, const double* head_decays,
                               void* o, void* block_states, int B, int T, int H, int dk, int dv, int block_size,
                               void* workspace, size_t workspace_bytes_given, void* stream) {
  const Shape s{B, T, H, dk, dv};
  const int segments = block_size >= 1 && check_shape(s, head_decays) == FP_OK ? plan_pop_forward(s, block_size) : 1;
  if (segments <= 1)
    return fp_pop_retention_fwd(q, k, v, s0, head_decays, o, block_states, B, T, H, dk, dv, block_size, stream);
  if (int rc = check_stream(stream, "fp_pop_retention_fwd_split")) return rc;
  if (!q || !k || !v || !o || !block_states) return fail(FP_ERR_NULL_POINTER, "q, k, v, o and block_states must not be NULL");
  if (int rc = check_workspace(s, segments, workspace, workspace_bytes_given, "fp_pop_retention_workspace_bytes")) return rc;
  return forward_split(s, block_segments(s, block_size), q, k, v, s0, head_decays, o, nullptr, workspace, stream,
                       BlockStates{out(block_states), nullptr, T / block_size});
}

int fp_pop_retention_bwd_split(const void* q, const void* k, const void* v, const void* s0, const double* head_decays,
                               const void* d_o, const void* d_block_states, void* dq, void* dk_, void* dv_, void* d_s0,
                               int B, int T, int H, int dk, int dv, int block_size, void* workspace,
                               size_t workspace_bytes_given, int forward_states_kept, void* stream) {
  const Shape s{B, T, H, dk, dv};
  const int segments = block_size >= 1 && check_shape(s, head_decays) == FP_OK ? plan_pop_backward(s, block_size) : 1;
  if (segments <= 1)
    return fp_pop_retention_bwd(q, k, v, s0, head_decays, d_o, d_block_states, dq, dk_, dv_, d_s0, B, T, H, dk, dv, block_size, stream);
  if (int rc = check_stream(stream, "fp_pop_retention_bwd_split")) return rc;
  if (!q || !k || !v || !d_o || !dq || !dk_ || !dv_)
    return fail(FP_ERR_NULL_POINTER, "q, k, v, d_o, dq, dk and dv must not be NULL");
  if (int rc = check_workspace(s, segments, workspace, workspace_bytes_given, "fp_pop_retention_workspace_bytes")) return rc;
  return backward_split(s, block_segments(s, block_size), q, k, v, s0, head_decays, d_o, nullptr, dq, dk_, dv_, d_s0, workspace,
                        forward_states_kept != 0, stream, BlockStates{nullptr, in(d_block_states), T / block_size});
}

int fp_pop_retention_bwd(const void* q, const void* k, const void* v, const void* s0, const double* head_decays,
                         const void* d_o, const void* d_block_states, void* dq, void* dk_, void* dv_, void* d_s0,
                         int B, int T, int H, int dk, int dv, int block_size, void* stream) {
  const Shape s{B, T, H, dk, dv};
  if (int rc = check_shape(s, head_decays)) return rc;
  if (int rc = check_stream(stream, "fp_pop_retention_bwd")) return rc;
  if (block_size < 1) return fail(FP_ERR_BAD_SHAPE, "block_size must be >= 1 (got %d)", block_size);
  if (!q || !k || !v || !d_o || !dq || !dk_ || !dv_)
    return fail(FP_ERR_NULL_POINTER, "q, k, v, d_o, dq, dk and dv must not be NULL");
  const void* d_blocks = (T / block_size > 0) ? d_block_states : nullptr;
  return backward(s, q, k, v, s0, head_decays, d_o, nullptr, d_blocks, block_size, dq, dk_, dv_, d_s0, stream);
}

int fp_pop_fused_fwd(const void* q, const void* k, const void* v, const void* s0, const void* q_sfx, const void* k_sfx,
                     const void* v_sfx, const double* head_decays, void* o, void* o_sfx, void* s_out, int B, int T,
                     int H, int dk, int dv, int block_size, int sfx_len, void* stream) {
  const Shape s{B, T, H, dk, dv};
  if (int rc = check_shape(s, head_decays)) return rc;
  if (int rc = check_stream(stream, "fp_pop_fused_fwd")) return rc;
  if (int rc = check_fused(s, block_size, sfx_len)) return rc;
  if (!q || !k || !v || !o || !q_sfx || !k_sfx || !v_sfx || !o_sfx)
    return fail(FP_ERR_NULL_POINTER, "q, k, v, o and their suffix counterparts must not be NULL");
  return fused_forward(s, q, k, v, s0, Suffixes{q_sfx, k_sfx, v_sfx, sfx_len}, head_decays, o, o_sfx, s_out, block_size,
                       stream);
}

int fp_pop_fused_bwd(const void* q, const void* k, const void* v, const void* s0, const void* q_sfx, const void* k_sfx,
                     const void* v_sfx, const double* head_decays, const void* d_o, const void* d_o_sfx,
                     const void* d_s_out, void* dq, void* dk_, void* dv_, void* dq_sfx, void* dk_sfx, void* dv_sfx,
                     void* d_s0, int B, int T, int H, int dk, int dv, int block_size, int sfx_len, void* stream) {
  const Shape s{B, T, H, dk, dv};
  if (int rc = check_shape(s, head_decays)) return rc;
  if (int rc = check_stream(stream, "fp_pop_fused_bwd")) return rc;
  if (int rc = check_fused(s, block_size, sfx_len)) return rc;
  if (!q || !k || !v || !q_sfx || !k_sfx || !v_sfx || !d_o || !d_o_sfx || !dq || !dk_ || !dv_ || !dq_sfx || !dk_sfx ||
      !dv_sfx)
    return fail(FP_ERR_NULL_POINTER, "inputs, d_o, d_o_sfx and the six gradient outputs must not be NULL");
  return fused_backward(s, q, k, v, s0, Suffixes{q_sfx, k_sfx, v_sfx, sfx_len}, head_decays, d_o, d_o_sfx, d_s_out, dq,
                        dk_, dv_, dq_sfx, dk_sfx, dv_sfx, d_s0, block_size, stream);
}

int fp_retention_decode_step(const void* q, const void* k, const void* v, const void* s_in, const double* head_decays,
                             void* o, void* s_out, int B, int H, int dk, int dv, void* stream) {
  const Shape s{B, 1, H, dk, dv};
  if (int rc = check_shape(s, head_decays)) return rc;
  if (!q || !k || !v || !o || !s_out) return fail(FP_ERR_NULL_POINTER, "q, k, v, o and s_out must not be NULL");
  fpk::DecodeArgs a;
  std::memset(&a, 0, sizeof a);
  a.q = in(q); a.k = in(k); a.v = in(v); a.s_in = in(s_in); a.s_out = out(s_out); a.o = out(o);
  a.B = B; a.H = H; a.dk = dk; a.dv = dv;
  a.scale = 1.0f / std::sqrt((float)dk);
  for (int h = 0; h < H; ++h) a.gamma[h] = (float)head_decays[h];
  const char* msg = "";
  if (fpk_launch_decode(a, stream, &msg) != 0) return fail(FP_ERR_LAUNCH, "decode step: %s", msg);
  return FP_OK;
}

int fp_rotary_qk(const void* q_in, const void* k_in, void* q_out, void* k_out, const float* theta, const long long* start,
                 long long start0, int B, int T, int H, int d, int inverse, void* stream) {
  if (!q_in || !q_out || !theta) return fail(FP_ERR_NULL_POINTER, "q_in, q_out and theta must not be NULL");
  if ((k_in == nullptr) != (k_out == nullptr)) return fail(FP_ERR_NULL_POINTER, "k_in and k_out must both be given or both be NULL");
  if (B < 1 || T < 1 || H < 1) return fail(FP_ERR_BAD_SHAPE, "B, T, H must be >= 1 (got %d, %d, %d)", B, T, H);
  if (d < 8 || d % 8 != 0) return fail(FP_ERR_UNSUPPORTED_DIM, "the head dimension must be a multiple of 8 (got %d)", d);
  if (misaligned(q_in) || misaligned(k_in) || misaligned(q_out) || misaligned(k_out))
    return fail(FP_ERR_BAD_SHAPE, "q and k must be 16-byte aligned");
  fpk::RotaryArgs a;
  std::memset(&a, 0, sizeof a);
  a.q_in = in(q_in); a.k_in = in(k_in); a.q_out = out(q_out); a.k_out = out(k_out);
  a.theta = theta; a.start = start; a.start0 = start0;
  a.B = B; a.T = T; a.H = H; a.d = d;
  a.sign = inverse ? -1.f : 1.f;
  const char* msg = "";
  if (fpk_launch_rotary(a, stream, &msg) != 0) return fail(FP_ERR_LAUNCH, "%s", msg);
  return FP_OK;
}

namespace {

int gated_norm(const void* r, const void* g, const void* d_out, void* y, void* d_r, void* d_g, long long rows, int H,
               int dv, double eps, void* stream) {
  if (rows < 1 || H < 1) return fail(FP_ERR_BAD_SHAPE, "rows and H must be >= 1 (got %lld, %d)", rows, H);
  const int lanes = dv / 8;
  if (dv < 8 || dv % 8 != 0 || lanes > 64 || (lanes & (lanes - 1)) != 0)
    return fail(FP_ERR_UNSUPPORTED_DIM, "dv must be 8 times a power of two, at most 512 (got %d)", dv);
  if (!(eps >= 0.0)) return fail(FP_ERR_BAD_SHAPE, "eps must be non-negative (got %g)", eps);
  if (misaligned(r) || misaligned(g) || misaligned(d_out) || misaligned(y) || misaligned(d_r) || misaligned(d_g))
    return fail(FP_ERR_BAD_SHAPE, "tensors must be 16-byte aligned");
  fpk::GatedNormArgs a;
  std::memset(&a, 0, sizeof a);
  a.r = in(r); a.g = in(g); a.d_out = in(d_out); a.out = out(y); a.d_r = out(d_r); a.d_g = out(d_g);
  a.groups = rows * H;
  a.dv = dv;
  a.eps = (float)eps;
  const char* msg = "";
  if (fpk_launch_gated_norm(a, stream, &msg) != 0) return fail(FP_ERR_LAUNCH, "%s", msg);
  return FP_OK;
}

}  // namespace

int fp_gated_group_norm_fwd(const void* r, const void* g, void* out_, long long rows, int H, int dv, double eps,
                            void* stream) {
  if (!r || !g || !out_) return fail(FP_ERR_NULL_POINTER, "r, g and out must not be NULL");
  return gated_norm(r, g, nullptr, out_, nullptr, nullptr, rows, H, dv, eps, stream);
}

int fp_gated_group_norm_bwd(const void* r, const void* g, const void* d_out, void* d_r, void* d_g, long long rows, int H,
                            int dv, double eps, void* stream) {
  if (!r || !g || !d_out || !d_r || !d_g) return fail(FP_ERR_NULL_POINTER, "r, g, d_out, d_r and d_g must not be NULL");
  return gated_norm(r, g, d_out, nullptr, d_r, d_g, rows, H, dv, eps, stream);
}

int fp_set_backward_choice(int choice, int checkpoint_every) {
  read_environment();
  if (choice < BWD_AUTO || choice > BWD_FUSED_PACED)
    return fail(FP_ERR_BAD_CONFIG, "backward choice %d: expected 0 (by shape), 1 (passes), 2 (fused) or 3 (fused, paced)", choice);
  if (checkpoint_every >= 0 && checkpoint_every % fpk::CH != 0)
    return fail(FP_ERR_BAD_CONFIG, "the checkpoint interval must be a multiple of %d tokens (got %d)", fpk::CH, checkpoint_every);
  g_bwd_choice.store(choice, std::memory_order_relaxed);
  if (checkpoint_every >= 0) g_ckpt_every.store(checkpoint_every, std::memory_order_relaxed);
  return FP_OK;
}

const char* fp_last_error(void) { return g_err; }

int fp_version(void) { return 1009; }

}  // extern "C"
