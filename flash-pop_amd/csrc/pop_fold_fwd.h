// Forward of a POP call with suffixes of at most 16 tokens and 64-wide keys (fp_pop_fused_fwd): the suffixes are part of the chunks
// that start at their boundaries, where the suffix walk of retention_pass_ws.h takes each of them as one more item.
//
//   o_i   = scale sum_{j <= i} gamma^(i-j) (q_i . k_j) v_j + gamma^(i+1) q_i S         S: the state at the chunk's start
//   o_s,i = the same inside the suffix, with the state at its boundary, which is the chunk's
//   S    <- gamma^L S + sum_j (scale gamma^(L-1-j) k_j)^T v_j
//
// One workgroup of 8 waves owns one (batch, head) stream and 64 columns of v, o and S and walks the chunks in order (64 tokens,
// cut at block boundaries; one more, empty, at T for the suffix there).  Waves w and w + 4 share a SIMD:
//
//   carry waves (0..3)  each a strip of 32 columns of S in fp32 accumulators and 32 of a chunk's rows (two waves hold the same
//                       strip).  The rows of a converted accumulator tile are put in such an order (`swapped`) that it is the
//                       read-out's operand as it is: S never goes through LDS.  First half of a step: the read-outs of q and
//                       q_s, the products with v, the outputs; second half: the state update, from registers.
//   feed waves (4..7)   loads (two chunks ahead), LDS tiles (one chunk ahead; k a second time, weighted for the update), the score
//                       tiles of the next chunk and of its suffix, the way out of the staged outputs.
//
// Two workgroup barriers per step.  What bounds it: the feed waves' chain, 1 100 cycles for the scores, 1 400 for the tiles, 600
// for the loads.  B8 H12 T2048 64 x 128, blocks of 64, suffixes of 16: forwards in a row 79.8 us each in the suffix walk (64 chunk
// items and 65 suffix items), 61.0 here; the launch in a traced training step 77.7 and 67.  128-wide keys were slower in it (B8 H16
// T4096: 230 against 190 us; both roles need more than 256 registers) and stay with the walk.
#pragma once
#include <type_traits>

#include "pass_args.h"
#include "lds_access.h"
#include "retention_bwd_fused.h"

namespace fpk {

constexpr int PF_DK = 64;          // columns of q and k
constexpr int PF_SFX = 16;         // longest suffix
constexpr int PF_FEED = 256;       // threads of each role
constexpr int PF_THREADS = 2 * PF_FEED;
constexpr int PF_LD = PF_DK + 8;   // row pitch of every tile, elements: 4 banks more than a multiple of 32
constexpr int PF_TILE = CH * PF_LD, PF_SFX_TILE = PF_SFX * PF_LD;
constexpr int PF_STAGE = 4 * PF_TILE + 3 * PF_SFX_TILE;   // q, k, k weighted, v; q_s, k_s, v_s
constexpr int PF_SCORES = 4 * FB_XP;                      // diagonal of row block 0, of row block 1, the tile below, the suffix's
constexpr int PF_IN_LD = BV + 4;                          // pitch of the state that enters, which takes the second set of score tiles and the staged outputs
constexpr int PF_OUT_LD = 40;                             // pitch of a wave's part of the state that leaves
constexpr int pf_lds_bytes() { return 2 * (2 * PF_STAGE + 2 * PF_SCORES + PF_TILE + PF_SFX_TILE); }
static_assert(PF_SCORES + PF_TILE + PF_SFX_TILE >= PF_DK * PF_IN_LD, "the state that enters fits");
static_assert(PF_DK == BV, "one tile shape for q, k and v");

namespace pf {

using namespace fb;

// Accumulator row / operand row m of a group of 16 stands for position 8 (bit 2) + 4 (bit 3) + (bits 0, 1): a lane then holds
// eight consecutive positions per k-step, which is a column-wise operand as it is.
FP_DEVICE int swapped(int m) { return (m & ~12) | ((m & 4) << 1) | ((m & 8) >> 1); }
// tr_lane with the columns of a group of 16 in that order
template <int LD>
FP_DEVICE TrLane tr_lane_swapped(int lane, TrOrder order) {
  return tr_lane<LD>((lane & ~3) | ((lane & 1) << 1) | ((lane & 2) >> 1), order);
}
FP_DEVICE u32x4 packed(const f32x16& v, int half) {
  u32x4 d;
#pragma unroll
  for (int e = 0; e < 4; ++e) d[e] = fprt::pack_bf16x2(v[8 * half + 2 * e], v[8 * half + 2 * e + 1]);
  return d;
}

}  // namespace pf

FP_DEVICE void pop_fold_fwd(const PassArgs& p, char* lds, int wg) {
  using namespace pf;
  constexpr int LD = PF_LD, KS = PF_DK / 16, NAB = PF_DK / 32;
  constexpr int PPR = PF_DK / 8, ROWS = PF_FEED / PPR, NU = CH / ROWS;   // 16-byte pieces per row, rows per sweep of a role, sweeps
  // stage s at base + s PF_STAGE
  uint16_t* const Qs = reinterpret_cast<uint16_t*>(lds);
  uint16_t* const Ks = Qs + PF_TILE;
  uint16_t* const Kw = Ks + PF_TILE;             // rows weighted for the state update
  uint16_t* const Vs = Kw + PF_TILE;
  uint16_t* const QsS = Vs + PF_TILE;
  uint16_t* const KsS = QsS + PF_SFX_TILE;
  uint16_t* const VsS = KsS + PF_SFX_TILE;
  // scores of the step it at base + (it & 1) PF_SCORES
  uint16_t* const XP = Qs + 2 * PF_STAGE;
  uint16_t* const OB = XP + 2 * PF_SCORES;       // staged o
  uint16_t* const OBS = OB + PF_TILE;            // staged o_s
  uint16_t* const IN = XP + PF_SCORES;

  const int tid = fprt::thread_index(), wave = tid >> 6, lane = tid & 63, g = lane >> 5, c = lane & 31;
  const int ntile = p.dB / BV;
  const int tile = wg % ntile, h = (wg / ntile) % p.H, b = (wg / ntile) / p.H;
  const float lg = p.log2g[h];
  const int bs = p.block, T = p.T;

  struct Chunk {
    int t0, L;
    bool ok;   // !ok: beyond the walk
    int sfx;   // the number of the suffix at its first token, -1: none
  };
  auto chunk_from = [&](int pos) {
    const int blk = pos / bs, nbnd = (blk + 1) * bs, end = pos + CH < nbnd ? pos + CH : nbnd;
    return Chunk{pos, pos < T ? end - pos : 0, true, pos == blk * bs ? blk : -1};
  };
  auto chunk_after = [&](const Chunk& k) { return k.ok && k.L > 0 ? chunk_from(k.t0 + k.L) : Chunk{0, 0, false, -1}; };
  const Chunk first = chunk_from(0);

  if (wave >= 4) {
    // ================================= feed waves =================================
    const int t = tid - PF_FEED, pw = wave - 4;
    const uint32_t rowA = (uint32_t)p.H * PF_DK * 2, rowB = (uint32_t)p.H * p.dB * 2;   // bytes between tokens
    const uint32_t headA = (uint32_t)h * PF_DK * 2, headB = ((uint32_t)h * p.dB + (uint32_t)tile * BV) * 2;
    auto view = [&](const void* base, uint32_t row, int rows, uint32_t pitch, uint32_t head) {
      return fprt::make_buf(static_cast<const char*>(base) + (size_t)row * pitch + head, rows > 0 ? (uint32_t)(rows - 1) * pitch + PF_DK * 2 : 0u);
    };
    auto ctx_row = [&](const Chunk& k) { return (uint32_t)b * T + k.t0; };
    auto sfx_row = [&](const Chunk& k) { return k.sfx >= 0 ? ((uint32_t)b * (p.nblk + 1) + k.sfx) * p.Ls : 0u; };
    auto sfx_rows = [&](const Chunk& k) { return k.sfx >= 0 ? p.Ls : 0; };
    // this thread's pieces: rows row + ROWS u (of a suffix: row, if there is one)
    const int row = t / PPR, col = 8 * (t % PPR), off = row * LD + col;
    const bool in_sfx = row < PF_SFX;
    struct Rows {
      u32x4 q[NU], k[NU], v[NU], qs, ks, vs;
    };
    auto load = [&](Rows& r, const Chunk& k) {
      const fprt::BufView qv = view(p.X, ctx_row(k), k.L, rowA, headA), kv = view(p.W, ctx_row(k), k.L, rowA, headA),
                          vv = view(p.Z, ctx_row(k), k.L, rowB, headB);
      const uint32_t oa = (uint32_t)row * rowA + col * 2, ob = (uint32_t)row * rowB + col * 2;
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        r.q[u] = fprt::buf_load128(qv, oa + (uint32_t)(ROWS * u) * rowA);
        r.k[u] = fprt::buf_load128(kv, oa + (uint32_t)(ROWS * u) * rowA);
        r.v[u] = fprt::buf_load128(vv, ob + (uint32_t)(ROWS * u) * rowB);
      }
      // (rows past the suffix are beyond the views)
      r.qs = fprt::buf_load128(view(p.Xs, sfx_row(k), sfx_rows(k), rowA, headA), oa);
      r.ks = fprt::buf_load128(view(p.Ws, sfx_row(k), sfx_rows(k), rowA, headA), oa);
      r.vs = fprt::buf_load128(view(p.Zs, sfx_row(k), sfx_rows(k), rowB, headB), ob);
    };
    auto stage = [&](const Rows& r, const Chunk& k, int s) {
      const int so = s * PF_STAGE + off;
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        const int o = so + ROWS * u * LD;
        st128(Qs + o, r.q[u]);
        st128(Ks + o, r.k[u]);
        st128(Vs + o, r.v[u]);
        const int left = k.L - 1 - row - ROWS * u;   // rows beyond a short chunk are zeros, their weight only has to be finite
        const float w = p.s_update * fprt::exp2_approx((float)(left > 0 ? left : 0) * lg);
        const float weights[8] = {w, w, w, w, w, w, w, w};
        st128(Kw + o, weigh(r.k[u], weights));
      }
      if (in_sfx) {
        st128(QsS + so, r.qs);
        st128(KsS + so, r.ks);
        st128(VsS + so, r.vs);
      }
    };
    auto drain = [&](const Chunk& k) {
      const fprt::BufView ov = view(p.Y, ctx_row(k), k.L, rowB, headB);
      const uint32_t ob = (uint32_t)row * rowB + col * 2;
#pragma unroll
      for (int u = 0; u < NU; ++u) fprt::buf_store128_nt(ov, ob + (uint32_t)(ROWS * u) * rowB, ld128(OB + off + ROWS * u * LD));
      if (in_sfx) fprt::buf_store128_nt(view(p.Ys, sfx_row(k), sfx_rows(k), rowB, headB), ob, ld128(OBS + off));
    };
    // Score tiles: the diagonal ones by feed waves 0 and 1, the one below by wave 2, the suffix's by wave 3.
    const bool diagonal = pw != 2;
    const int s_ib = pw == 0 ? 0 : 1, s_jb = pw == 1 ? 1 : 0;   // rows of q, rows of k
    float mw[16];
    score_weights(p.s_intra, lg, diagonal, false, c, g, mw);
    const uint16_t* const xrow = pw == 3 ? QsS + (c & (PF_SFX - 1)) * LD + 8 * g : Qs + (32 * s_ib + c) * LD + 8 * g;
    const uint16_t* const wrow = pw == 3 ? KsS + (score_row(c) & (PF_SFX - 1)) * LD + 8 * g : Ks + (32 * s_jb + score_row(c)) * LD + 8 * g;
    uint16_t* const xp = XP + (pw == 3 ? 3 : diagonal ? s_ib : 2) * FB_XP;
    auto scores = [&](int s) {
      u32x4 xf[KS], wf[KS];
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        xf[k] = frag_cols(xrow + s * PF_STAGE, k);
        wf[k] = frag_cols(wrow + s * PF_STAGE, k);
      }
      fprt::sched_fence();
      f32x16 sc = {0};
#pragma unroll
      for (int k = 0; k < KS; ++k) sc = fprt::mfma_32x32x16_bf16(wf[k], xf[k], sc);
      score_finish(sc, mw, diagonal, false, c, g, xp + s * PF_SCORES, lane);
    };

    Chunk c0 = first, c1 = chunk_after(c0), c2 = chunk_after(c1), c3 = chunk_after(c2);
    Rows ra, rb;
    // (the fences keep the order of the loads, on which the counts of those still to come depend)
    load(ra, c0);
    fprt::sched_fence();
    load(rb, c1);
    fprt::sched_fence();
    stage(ra, c0, 0);
    fprt::sched_fence();
    load(ra, c2);
    fprt::sched_fence();
    stage(rb, c1, 1);
    fprt::sched_fence();
    load(rb, c3);
    fprt::sched_fence();
    fprt::block_sync();
    scores(0);
    fprt::block_sync();
    // c0 is being worked on, c1 is in LDS, c2 and c3 are on their way
    auto step = [&](Rows& r, int s) {
      scores(s ^ 1);
      fprt::block_sync();
      const Chunk done = c0;
      fprt::sched_fence();
      stage(r, c2, s);
      const Chunk c4 = chunk_after(c3);
      fprt::sched_fence();
      load(r, c4);
      fprt::sched_fence();
      drain(done);
      fprt::sched_fence();
      c0 = c1; c1 = c2; c2 = c3; c3 = c4;
      fprt::block_sync();
      return c0.ok;
    };
    while (step(ra, 0) && step(rb, 1)) {}
    return;
  }

  // ================================= carry waves =================================
  const int ns = wave & 1, ih = wave >> 1;      // this wave: columns 32 ns .., chunk rows 32 ih ..
  // racc[a] element r is S[32 a + 16 (r / 8) + 8 g + r % 8][n], n = 32 ns + swapped(c)
  f32x16 racc[NAB];
  const size_t matrix = ((size_t)b * p.H + h) * PF_DK * p.dB;
  const uint32_t mat_bytes = (uint32_t)(PF_DK * p.dB * 2);
  if (p.R0) {
    const fprt::BufView v = fprt::make_buf(p.R0 + matrix, mat_bytes);
    constexpr int NP = PF_DK * PPR / PF_FEED;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int q = tid + PF_FEED * i;
      const u32x4 m = fprt::buf_load128(v, ((uint32_t)(q / PPR) * p.dB + tile * BV + 8 * (q % PPR)) * 2);
      uint16_t* const d = IN + (q / PPR) * PF_IN_LD + 8 * (q % PPR);
      st64(d, u32x2{m[0], m[1]});
      st64(d + 4, u32x2{m[2], m[3]});
    }
  }
  fprt::block_sync();
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    u32x4 u = {0, 0, 0, 0};
    if (p.R0) u = frag_rows<PF_IN_LD>(IN, tr_lane_swapped<PF_IN_LD>(lane, TR_SEQ), s, 32 * ns);
#pragma unroll
    for (int e = 0; e < 8; ++e) racc[s >> 1][8 * (s & 1) + e] = bf16_elem(u, e);
  }
  fprt::block_sync();

  const TrLane tr = tr_lane_swapped<LD>(lane, TR_ACC), tr_nat = tr_lane_swapped<LD>(lane, TR_NAT);
  const uint16_t* const xrow = Qs + (32 * ih + c) * LD + 8 * g;
  const uint16_t* const xsrow = QsS + (c & (PF_SFX - 1)) * LD + 8 * g;
  const float wread = p.s_read * fprt::exp2_approx((float)(32 * ih + c + 1) * lg), wread_sfx = p.s_read * fprt::exp2_approx((float)(c + 1) * lg);
  const float gL_full = fprt::exp2_approx((float)CH * lg);

  Chunk cur = first;
  auto step = [&](int s) {
    const int L = cur.L, so = s * PF_STAGE;
    const bool has_sfx = ih == 0 && cur.sfx >= 0;
    const uint16_t* const xps = XP + s * PF_SCORES + lane * 8;

    // ---- first half: everything that reads the chunk's tiles, and the outputs
    u32x4 xf[KS], qf[KS], zi[2], zj[2], zs = {0, 0, 0, 0}, pi[2], pj[2], ps = {0, 0, 0, 0};
    u32x4 zw[4], wa[4][NAB];
#pragma unroll
    for (int k = 0; k < KS; ++k) xf[k] = frag_cols(xrow + so, k);
    if (has_sfx) {
#pragma unroll
      for (int k = 0; k < KS; ++k) qf[k] = frag_cols(xsrow + so, k);
      zs = frag_rows<LD>(VsS + so, tr, 0, 32 * ns);
      ps = ld128(xps + 3 * FB_XP);
    }
    // v of this row block's tokens and of the other block's, the latter for the rows that come after them
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      zi[k] = frag_rows<LD>(Vs + so + 32 * ih * LD, tr, k, 32 * ns);
      pi[k] = ld128(xps + ih * FB_XP + 512 * k);
      zj[k] = frag_rows<LD>(Vs + so + 32 * (1 - ih) * LD, tr, k, 32 * ns);
      pj[k] = ld128(xps + 2 * FB_XP + 512 * k);
    }
    fprt::sched_fence();
    f32x16 acc = {0}, accs = {0};
#pragma unroll
    for (int k = 0; k < KS; ++k) {   // (q S)^T[n][i] = sum_a S[a][n] q[i][a]
      const u32x4 ra = packed(racc[k >> 1], k & 1);
      acc = fprt::mfma_32x32x16_bf16(ra, xf[k], acc);
      if (has_sfx) accs = fprt::mfma_32x32x16_bf16(ra, qf[k], accs);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      zw[k] = frag_rows<LD>(Vs + so, tr_nat, k, 32 * ns);
#pragma unroll
      for (int a = 0; a < NAB; ++a) wa[k][a] = frag_rows<LD>(Kw + so, tr_nat, k, 32 * a);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] *= wread;
#pragma unroll
    for (int k = 0; k < 2; ++k) acc = fprt::mfma_32x32x16_bf16(zi[k], pi[k], acc);
    if (ih == 1) {
#pragma unroll
      for (int k = 0; k < 2; ++k) acc = fprt::mfma_32x32x16_bf16(zj[k], pj[k], acc);
    }
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) st128(OB + (32 * ih + c) * LD + 32 * ns + 16 * hf + 8 * g, packed(acc, hf));
    if (has_sfx) {
#pragma unroll
      for (int r = 0; r < 16; ++r) accs[r] *= wread_sfx;
      accs = fprt::mfma_32x32x16_bf16(zs, ps, accs);
      if (c < PF_SFX) {
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) st128(OBS + c * LD + 32 * ns + 16 * hf + 8 * g, packed(accs, hf));
      }
    }
    fprt::block_sync();

    // ---- second half: the state update, from registers
    const float gL = L == CH ? gL_full : fprt::exp2_approx((float)L * lg);
#pragma unroll
    for (int a = 0; a < NAB; ++a) {
#pragma unroll
      for (int r = 0; r < 16; ++r) racc[a][r] *= gL;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
#pragma unroll
      for (int a = 0; a < NAB; ++a) racc[a] = fprt::mfma_32x32x16_bf16(wa[k][a], zw[k], racc[a]);
    }
    cur = chunk_after(cur);
    fprt::block_sync();
    return cur.ok;
  };
  while (step(0) && step(1)) {}

  // The state at T: a 32-row block of the strip per wave, through a piece of the tiles that only this wave uses now
  if (p.Rout) {
    const fprt::BufView v = fprt::make_buf(p.Rout + matrix, mat_bytes);
    uint16_t* const st = Qs + wave * 32 * PF_OUT_LD;
    auto store = [&](int a, const f32x16& acc) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        reinterpret_cast<u16_m*>(st)[(16 * (r >> 3) + 8 * g + (r & 7)) * PF_OUT_LD + swapped(c)] = float_to_bf16_bits(acc[r]);
      fprt::wave_sync();
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int row = (lane >> 2) + 16 * i, piece = lane & 3;
        fprt::buf_store128(v, ((uint32_t)(32 * a + row) * p.dB + tile * BV + 32 * ns + 8 * piece) * 2, ld128(st + row * PF_OUT_LD + 8 * piece));
      }
    };
    if (ih == 0) store(0, racc[0]);
    else store(1, racc[1]);
  }
}

// Whether the kernel above takes a planned pass on a device of `compute_units`: a forward with suffixes that fit beside a chunk,
// keys of 64, whole blocks of at most a chunk and a half or so, where it is the faster one.  Its step takes about 1.7 us against 1.1 for
// an item of the walk, and a workgroup half a microsecond longer to start, so it needs enough suffixes to save, and of 64 x 64
// states on a full device, where the bytes count too, more of them (512 a token and tile; 384 at 64 x 128, 320 at 64 x 256).
// Speed here over that of the walk, inputs not in a cache, 128 to 1 024 workgroups, blocks of 16 to 64 tokens:
//                1 block        2 blocks       3 blocks       4 blocks       6 blocks       12 blocks      32 blocks
//   64 x 64      .79 to .94     .84 to 1.02    .89 to 1.07    .93 to 1.11    .94 to 1.18    1.01 to 1.29   1.08 to 1.41
//   64 x 128     .85 to .92     .90 to 1.00    .97 to 1.06    1.01 to 1.11   1.02 to 1.20   1.09 to 1.30   1.13 to 1.41
//   64 x 256     .85 to .95     .93 to 1.00    .97 to 1.08    1.03 to 1.13   1.06 to 1.19   1.09 to 1.30   1.10 to 1.40
// (the longer the block the lower; 32 workgroups of 64 x 64: 4 blocks of 64 1.08, 6 blocks 1.13), blocks of 72 to 96, 104 and 128:
//                4 blocks                          8 blocks                           12 blocks
//   64 x 64      .95 to 1.00, .92 to .99, .90      .99 to 1.06, .95 to 1.03, .89      1.01 to 1.08, .97 to 1.04, .93 to 1.00
//   64 x 128     .97 to 1.00, .97 to 1.00, .92     1.02 to 1.07, 1.01 to 1.06, .89    1.03 to 1.09, 1.02 to 1.08, .94 to 1.03
//   64 x 256     .98 to 1.02, .99 to 1.00, .93     1.02 to 1.06, 1.01 to 1.06, .94    1.03 to 1.09, 1.03 to 1.08, .94 to 1.05
inline bool pop_folds(const PassArgs& a, int compute_units) {
  if (a.Ls <= 0 || a.Ls > PF_SFX || a.reverse || a.dA != PF_DK || a.T != a.nblk * a.block || a.rs_n != 1) return false;
  const bool by_bytes = a.dB == BV && 2LL * a.B * a.H > compute_units;
  if (a.block > CH) return a.block <= (a.dB == BV ? 96 : 104) && a.nblk >= (by_bytes ? 12 : 8);
  if (by_bytes) return a.nblk >= 3 && 4 * a.nblk >= a.block - 16;
  return a.nblk >= (2 * a.block <= CH ? 3 : 4);
}

}  // namespace fpk
