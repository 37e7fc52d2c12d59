// State-only pass for states of 64 or 128 rows: what a sequence (of any length) adds to the
// carried state when nothing else is wanted of the pass (the first step of the split-sequence path),
//   U[a][n] = sum over the tokens j of  weight(j) W[j][a] Z[j][n],
// chunk by chunk as R <- gamma^64 R + (wkey W)^T Z from R = 0, with wkey(j) = s_update gamma^(63 - j)
// walking forward (gamma^(L - 1 - j) in a last chunk of L tokens) and s_update gamma^(j + 1) walking backward, the weighted W rounded to bf16 as the
// pass kernel rounds it.
//
// One workgroup per (sequence, head, NC columns of Z) holds its whole tile of R in the accumulators
// of its waves, so W is read once per NC columns, Z once, and nothing else moves.  The W and Z tiles
// of a chunk sit row-major in LDS (two stages) and both MFMA operands come from them through the
// transposing LDS read (the tile layout and the operand helpers are those of retention_bwd_fused.h);
// two more chunks are on their way in registers.  One workgroup barrier per chunk.
//
// 64 rows: 64 columns per workgroup of 256 threads (37 KB of LDS: several share a compute unit), bit for bit what the pass
// kernel's state-only walk gives, which takes all other states and many short sequences of these (contrib_pays):
// chunks are cut from where the walk starts, so that walking backward the short one is the first of the sequence, every weight is
// a power of gamma of its own, and the tokens are summed in order (ContribTile::AS_WALK).  64 x 128, B20 T256 H12 11.5 us in the
// walk, 8.8 here; B40 T128 H4 8.0, 6.2.  128 columns of a 64-row state per workgroup were slower.
//
// 128 rows: 128 columns per workgroup of 512 threads; chunks from the first token on in both directions, weights of a k-step
// from those of the one before.
//
// The sum leaves in whole lines: a lane holds eight consecutive columns of a row, which go through a row-major LDS tile (16 bits at a time
// it took as long as four chunks: 128 x 128, B12 T448 H8 17.1 -> 11.5 us a launch; in pieces of 32 bytes, through the transposing read, which
// took a second round for the lower halves, the launch of B1 H16 T1152 128 x 128 in segments of 4, 4, 4, 4 and 2 chunks took 11.5 us, so
// 10.0, written through 9.4; of equal segments, T1280, 8.1 -> 7.4; the forward of B2 H8 T1152 128 x 256 29.4 -> 27.4).
#pragma once
#include <type_traits>

#include "pass_args.h"
#include "lds_access.h"
#include "retention_bwd_fused.h"

namespace fpk {

// One workgroup's share: DK rows and NC columns of the state, NTH threads
template <int DK, int NC, int NTH>
struct ContribTile {
  static constexpr int LDW = DK + 8, LDZ = NC + 8;
  static constexpr int W = CH * LDW, STAGE = W + CH * LDZ;              // elements
  static constexpr int NRT = DK / 32, TPW = NRT * (NC / 32) / (NTH / 64);   // 32-row blocks of R; 32 x 32 tiles of it per wave
  static constexpr int NW = CH * (DK / 8) / NTH, NZ = CH * (NC / 8) / NTH;  // 16-byte pieces per thread
  static constexpr bool AS_WALK = NC == BV;
  // two stages of a W and a Z tile; R on its way out (both halves of it) takes their place
  static constexpr int lds_bytes = 2 * 2 * STAGE;
  static_assert(2 * STAGE >= 2 * DK * LDZ, "both halves of R fit where the tiles were");
  static_assert(NRT * (NC / 32) % (NTH / 64) == 0 && (NTH / 64) % NRT == 0, "whole tiles per wave");
};

// Row m of a group of 16 of an accumulator tile stands for column 8 (bit 2) + 4 (bit 3) + (bits 0, 1) of R: a lane then holds eight
// consecutive columns of a row.  The Z operand is read in that order: the pieces of four columns change places.
template <int LD>
FP_DEVICE fb::TrLane swapped_columns(int lane) {
  const fb::TrLane tr = fb::tr_lane<LD>(lane, fb::TR_NAT);
  const int piece = lane & 3, moved = 4 * ((((piece & 1) << 1) | (piece >> 1)) - piece);
  return fb::TrLane{tr.lo + moved, tr.hi + moved};
}
// 16 bits of each element of R (the tiles of this wave) -> the row-major LDS tile Rt, `column`: this lane's first
template <int TPW, int LD, typename Part>
FP_DEVICE void lay_contribution(uint16_t* Rt, int row, int column, const f32x16 (&racc)[TPW], Part part) {
#pragma unroll
  for (int u = 0; u < TPW; ++u) {
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      u32x4 d;
#pragma unroll
      for (int e = 0; e < 4; ++e) d[e] = pack16(racc[u][8 * hf + 2 * e], racc[u][8 * hf + 2 * e + 1], part);
      st128(Rt + fb::at<LD>(row, column + 32 * u + 16 * hf), d);
    }
  }
}

// AS_WALK: row r of a tile holds token `walk_in_row(r)`, so that element e of a TR_NAT operand is token walk_token(g, e) of its
// k-step, as in the pass kernel's operands.  (The threads fetch by that order and store row by row: with the rows' places permuted
// at the stores instead, the rows of a wave meet in the same banks.)
FP_DEVICE int walk_in_row(int r) { return (r & ~15) | ((r >> 2) & 3) | ((r & 2) << 1) | ((r & 1) << 3); }
FP_DEVICE int walk_token(int g, int e) { return 4 * g + (e & 3) + 8 * (e >> 2); }

template <int DK, int NC, int NTH, bool REV>
FP_DEVICE void segment_contrib(const ContribArgs& p, char* lds) {
  using namespace fb;
  using G = ContribTile<DK, NC, NTH>;
  constexpr int LDW = G::LDW, LDZ = G::LDZ, TPW = G::TPW;
  constexpr bool AS_WALK = G::AS_WALK;
  const int tid = fprt::thread_index(), wave = tid >> 6, lane = tid & 63, g = lane >> 5, c = lane & 31;
  // the workgroups of one (sequence, head) differ by a multiple of the stream count: with a multiple
  // of 8 streams they sit on the same XCD and share the W rows in its L2
  const int streams = p.B * p.H;
  const int ct = fprt::block_index() / streams, stream = fprt::block_index() % streams;
  const int h = stream % p.H, b = stream / p.H;
  // tokens of this sequence and its first row
  const int seg = p.segs > 0 ? b % p.segs : 0;
  const int len = p.segs > 0 && p.total - seg * p.T < p.T ? p.total - seg * p.T : p.T;
  const size_t row0 = p.segs > 0 ? (size_t)(b / p.segs) * p.total + (size_t)seg * p.T : (size_t)b * p.T;
  const int nch = (len + CH - 1) / CH;
  const float lg = p.log2g[h];
  const uint32_t roww = (uint32_t)p.H * DK * 2, rowz = (uint32_t)p.H * p.dB * 2;   // bytes between tokens
  const char* const wbase = reinterpret_cast<const char*>(p.W) + (row0 * p.H + h) * DK * 2;
  const char* const zbase = reinterpret_cast<const char*>(p.Z) + (row0 * p.H + h) * p.dB * 2 + (size_t)ct * NC * 2;

  uint16_t* const TL = reinterpret_cast<uint16_t*>(lds);   // stage s: W tile at s G::STAGE, Z tile behind it
  // this thread's 16-byte pieces: rows w_row + RW u of W, z_row + RZ u of Z
  constexpr int RW = NTH / (DK / 8), RZ = NTH / (NC / 8);
  const int w_place = tid / (DK / 8), w_piece = tid % (DK / 8), z_place = tid / (NC / 8), z_piece = tid % (NC / 8);
  const int w_off = at<LDW>(w_place, 8 * w_piece), z_off = at<LDZ>(z_place, 8 * z_piece);
  const int w_row = AS_WALK ? walk_in_row(w_place) : w_place, z_row = AS_WALK ? walk_in_row(z_place) : z_place;
  static_assert(RW % 16 == 0 && RZ % 16 == 0, "a thread's rows have the same place in their k-steps");
  struct Rows {
    u32x4 w[G::NW], z[G::NZ];
  };

  // registers <- the chunk visited it-th
  auto load = [&](int it, Rows& pf) {
    const bool live = it < nch;
    const int end = AS_WALK && REV ? len - it * CH : len;
    const int first = !(AS_WALK && REV) ? (REV ? nch - 1 - it : it) * CH : end > CH ? end - CH : 0;
    // rows of a short chunk from `end` on read as zeros (contrib_fits); visits beyond the walk read zeros and move nothing.  (One row
    // offset for all of a thread's loads: chosen per load, the choice became branches around them, behind which every wait is for all.)
    const fprt::BufView w = fprt::make_buf(wbase, live ? (uint32_t)(end - 1) * roww + DK * 2 : 0u);
    const fprt::BufView z = fprt::make_buf(zbase, live ? (uint32_t)(end - 1) * rowz + NC * 2 : 0u);
    const uint32_t t0 = live ? first : 0;
    const uint32_t wo = (t0 + w_row) * roww + w_piece * 16, zo = (t0 + z_row) * rowz + z_piece * 16;
#pragma unroll
    for (int u = 0; u < G::NW; ++u) pf.w[u] = fprt::buf_load128(w, wo + (uint32_t)(RW * u) * roww);
#pragma unroll
    for (int u = 0; u < G::NZ; ++u) pf.z[u] = fprt::buf_load128(z, zo + (uint32_t)(RZ * u) * rowz);
  };
  auto stage = [&](int s, const Rows& pf) {
    uint16_t* const st = TL + s * G::STAGE;
#pragma unroll
    for (int u = 0; u < G::NW; ++u) st128(st + w_off + RW * u * LDW, pf.w[u]);
#pragma unroll
    for (int u = 0; u < G::NZ; ++u) st128(st + G::W + z_off + RZ * u * LDZ, pf.z[u]);
  };

  Rows pa, pb;   // the first two chunks travel while the weights are made
  load(0, pa);
  load(1, pb);
  fprt::sched_fence();

  // this wave's tiles of R: rows a = 32 at_ .., columns n = 32 (nt0 + u) .., u < TPW
  const int at_ = wave % G::NRT, nt0 = (wave / G::NRT) * TPW;
  const TrLane tr_w = tr_lane<LDW>(lane, TR_NAT), tr_z = swapped_columns<LDZ>(lane);
  auto weight = [&](int e) { return p.s_update * fprt::exp2_approx((float)(e > 0 ? e : 0) * lg); };
  // Weights of a whole chunk.  AS_WALK: of every k-step.  Else of the k-step taken first (the last 16 tokens walking forward, the
  // first 16 walking backward); each further k-step is 16 tokens further from where the state is read.
  constexpr int NWK = AS_WALK ? 4 : 1;
  float wk_whole[NWK][8];
#pragma unroll
  for (int t = 0; t < NWK; ++t) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int j = AS_WALK ? 16 * t + walk_token(g, e) : REV ? nat_token(g, e) : 48 + nat_token(g, e);
      wk_whole[t][e] = p.s_update * fprt::exp2_approx((float)(REV ? j + 1 : CH - 1 - j) * lg);
    }
  }
  const float g16 = fprt::exp2_approx(16.f * lg), gL = fprt::exp2_approx((float)CH * lg);

  f32x16 racc[TPW];
#pragma unroll
  for (int u = 0; u < TPW; ++u) racc[u] = f32x16{0};

  // L: tokens of the chunk.  The short one that ends a walk forward (SHORT) has weights of its own, which count from its last
  // token, as in the walk that carries a sequence through, so that a cut call gives the state of the uncut one.  Walking backward
  // the weights are those of any other chunk, and with 128 columns the short chunk is met first, with R = 0.
  auto update = [&](int s, auto short_chunk, int L) {
    constexpr bool SHORT = decltype(short_chunk)::value;
    const uint16_t* const Ws = TL + s * G::STAGE;
    const uint16_t* const Zs = Ws + G::W;
    const float decay = SHORT || (AS_WALK && REV) ? fprt::exp2_approx((float)L * lg) : gL;
    u32x4 ua[4], ub[4][TPW];
    auto request = [&](int tt) {
      const int t = AS_WALK || REV ? tt : 3 - tt;
      ua[tt] = frag_rows<LDW>(Ws, tr_w, t, 32 * at_);
#pragma unroll
      for (int u = 0; u < TPW; ++u) ub[tt][u] = frag_rows<LDZ>(Zs, tr_z, t, 32 * (nt0 + u));
    };
    request(0);
    request(1);
    fprt::sched_fence();
#pragma unroll
    for (int u = 0; u < TPW; ++u) {
#pragma unroll
      for (int r = 0; r < 16; ++r) racc[u][r] *= decay;
    }
    float wk[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) wk[e] = wk_whole[0][e];
    fprt::sched_fence();
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) {
      if (SHORT) {
#pragma unroll
        for (int e = 0; e < 8; ++e) wk[e] = weight(L - 1 - (AS_WALK ? 16 * tt + walk_token(g, e) : 16 * (3 - tt) + nat_token(g, e)));
      } else if (AS_WALK) {
#pragma unroll
        for (int e = 0; e < 8; ++e) wk[e] = wk_whole[AS_WALK ? tt : 0][e];
      }
      const u32x4 wa = weigh(ua[tt], wk);
#pragma unroll
      for (int u = 0; u < TPW; ++u) racc[u] = fprt::mfma_32x32x16_bf16(ub[tt][u], wa, racc[u]);
      if (tt + 2 < 4) request(tt + 2);
      if (!AS_WALK && tt < 3) {
#pragma unroll
        for (int e = 0; e < 8; ++e) wk[e] *= g16;
      }
      fprt::sched_fence();
    }
  };

  // Chunk it is multiplied from stage it & 1 while chunk it + 1 moves from registers into the
  // other stage and the loads of chunk it + 3 take its place; chunk it + 2 is on its way in the
  // second set of registers.
  const int nwhole = REV ? nch : len / CH;
  auto tokens = [&](int it) { return AS_WALK && REV && len - it * CH < CH ? len - it * CH : CH; };
  stage(0, pa);
  load(2, pa);
  fprt::block_sync();
  for (int it = 0; it < nwhole; it += 2) {
    stage(1, pb);
    load(it + 3, pb);
    update(0, std::false_type{}, tokens(it));
    fprt::block_sync();
    if (it + 1 >= nwhole) break;
    stage(0, pa);
    load(it + 4, pa);
    update(1, std::false_type{}, tokens(it + 1));
    fprt::block_sync();
  }
  // (pb is wanted on both ways out of the loop, or the compiler moves its loads behind the break, a chunk later: 42 -> 46 us at
  // B2 H8 T16384 dv 256)
#pragma unroll
  for (int u = 0; u < G::NW; ++u) fprt::keep(pb.w[u]);
#pragma unroll
  for (int u = 0; u < G::NZ; ++u) fprt::keep(pb.z[u]);
  if (nwhole < nch) {
    update(nwhole & 1, std::true_type{}, len - nwhole * CH);
    fprt::block_sync();
  }

  // R -> its columns of the rows of U[b][h] (element (a, n) at a * dB + n), as bf16 or in fp32 halves, in whole lines through LDS; every
  // read of the tiles is behind the last barrier
  uint16_t* const lower = TL + DK * LDZ;
  const int row = 32 * at_ + c, column = 32 * nt0 + 8 * g;
  if (p.U_lo) {
    lay_contribution<TPW, LDZ>(TL, row, column, racc, UpperHalf{});
    lay_contribution<TPW, LDZ>(lower, row, column, racc, LowerHalf{});
  } else {
    lay_contribution<TPW, LDZ>(TL, row, column, racc, AsBf16{});
  }
  fprt::block_sync();
  const size_t matrix = (size_t)stream * DK * p.dB + (size_t)ct * NC;
  // Written through from 2 MB a plane on (then and written back at the kernel's end, whole calls, us): B1 H16 T2001 128 x 128, 2.6 MB,
  // 27.1 and 27.4; B1 H12 T5003 64 x 128, 3.9 MB, 28.2 and 28.8; below, B1 H4 T2048 64 x 64, .25 MB, 15.5 and 15.3, T4129 18.7 and 18.3.
  const bool through = (size_t)p.B * p.H * DK * p.dB * 2 >= (2u << 20);
  auto put = [&](uint16_t* dst, const uint16_t* Rt) {
    const fprt::BufView uv = fprt::make_buf(dst + matrix, (uint32_t)(DK - 1) * p.dB * 2 + NC * 2);
#pragma unroll
    for (int i = 0; i < DK * (NC / 8) / NTH; ++i) {
      const uint32_t to = (uint32_t)(z_place + RZ * i) * p.dB * 2 + z_piece * 16;
      const u32x4 d = ld128(Rt + z_off + RZ * i * LDZ);
      if (through) fprt::buf_store128_through(uv, to, d);
      else fprt::buf_store128(uv, to, d);
    }
  };
  put(p.U, TL);
  if (p.U_lo) put(p.U_lo, lower);
}

// Host side, shared by the GPU launcher and the CPU test harness: argument check.
inline const char* check_contrib(const ContribArgs& a) {
  if (a.B < 1 || a.T < 1 || a.H < 1 || a.H > MAX_HEADS) return "state-only pass: B, T, H >= 1 expected";
  if (a.segs < 0 || (a.segs > 0 && (a.B % a.segs != 0 || a.total > (long long)a.segs * a.T || a.total <= (a.segs - 1LL) * a.T)))
    return "state-only pass: segments that do not cover their sequence";
  if ((a.dk != 64 && a.dk != FB_D) || a.dB < a.dk || a.dB % a.dk != 0) return "state-only pass: W of 64 or 128 columns, Z of a multiple of them";
  if (!a.W || !a.Z || !a.U) return "state-only pass: null pointer";
  if (!contrib_fits(a.T, a.H, a.dk, a.dB)) return "state-only pass: sequence too long";
  if ((long long)a.B * a.H * (a.dB / a.dk) > 0x7fffffffLL) return "state-only pass: too many sequences";
  return nullptr;
}

}  // namespace fpk
