// Retention pass (see pass_args.h for the recurrence) with 128 columns of Z, Y and R per workgroup and dA = 128: one sequence (or
// segment) per workgroup, no block states, no suffixes.  Rows go from global memory into LDS as in retention_pass_fill.h, whose
// tiles, operand orders and one barrier per step these are, but a step is half of a 64-token chunk:
//
//   half 0 of a chunk (rows 0 .. 31; walking backward rows 32 .. 63)   the rest, half 1
//
//   carry waves (0..3)  each 32 columns of R and all rows of a half.  The converted R that the chunk starts with is the read-out's
//                       operand for both halves; decayed once, R then takes the rows of half 0 and of half 1.
//   feed waves  (4..7)  a half ahead of them: 4 makes the half's own score tile, 5 that of half 1 with the tokens of half 0, 6 and 7
//                       weigh W; 5, 6 and 7 copy the later rows of W, X and Z, 4 and 5 store the half before.
//
// Nothing is computed twice: 38 products a carry wave and chunk, where two workgroups of 64 columns make 28 each and every strip is held
// by two waves; X and W leave the L2 once per 128 columns; half-sized steps keep two to three of them on their way.
//
// What bounds it: from half of the device on the memory (B16 T2048 H8 128 x 256: 82 us, 55 with the copies alone, 402 MB in all), with
// few workgroups the feed waves' chain (1.15 us a chunk, the carry waves' 1.07, together 1.5; 1.8 with every copy, store and weight
// spread over all four).  The same pass by workgroups of 64 columns (retention_pass_ws.h): 115 us.  Both sides stand at pass_is_wide.
#pragma once
#include <type_traits>

#include "pass_args.h"
#include "lds_access.h"
#include "retention_pass_fill.h"

namespace fpk {

constexpr int PW_THREADS = 512;
constexpr int PW_D = 128;                  // columns of X and W, columns of Z, Y and R per workgroup
constexpr int PW_AHEAD = 4;                // halves between the step that asks for a half's rows and the one that carries it
constexpr int PW_ROWS = CH / 2;
constexpr int PW_PITCH = 2 * PW_D;
constexpr int PW_TILE = PW_ROWS * PW_PITCH;
constexpr int pw_lds_bytes() {
  return PW_AHEAD * PW_TILE               // X
         + 2 * (PW_AHEAD + 1) * PW_TILE   // W, Z
         + 2 * PW_TILE                    // W weighted
         + 2 * 2 * FP_P                   // scores: own tile, other tile
         + 2 * 4 * FP_Q;                  // staged output
}

template <bool REV>
FP_DEVICE void retention_pass_wide_dir(const PassArgs& p, const PassTensors& io, char* lds, int wg) {
  using namespace pp;
  constexpr int DA = PW_D, AHEAD = PW_AHEAD, KS = DA / 16, NAB = DA / 32, COPIES = 8;   // of a wave that copies, per step
  constexpr int X0 = 0, W0 = X0 + AHEAD * PW_TILE, Z0 = W0 + (AHEAD + 1) * PW_TILE, WW0 = Z0 + (AHEAD + 1) * PW_TILE, P0 = WW0 + 2 * PW_TILE,
                Q0 = P0 + 2 * 2 * FP_P;
  auto at = [&](int byte) { return reinterpret_cast<uint16_t*>(lds + byte); };
  auto key = [](int row) { return ((row & 3) << 2) | ((row >> 2) & 3); };
  auto place = [&](int row, int piece) { return row * PW_PITCH + 16 * (piece ^ key(row)); };
  // the stage after one that starts `off` bytes into the ring of X, into those of W and Z
  auto next_x = [](int off) { return off == (AHEAD - 1) * PW_TILE ? 0 : off + PW_TILE; };
  auto next_w = [](int off) { return off == AHEAD * PW_TILE ? 0 : off + PW_TILE; };

  const int tid = fprt::thread_index(), wave = (int)fprt::uniform((uint32_t)tid >> 6), lane = tid & 63, g = lane >> 5, c = lane & 31;
  const int ntile = p.dB / PW_D;
  const int tile = wg % ntile, h = (wg / ntile) % p.H, slot = (wg / ntile) / p.H;
  const float lg = p.log2g[h];
  const ChunkWalk<FILL_PLAIN, REV> walk{p};
  // A half of a chunk: its first row in the chunk, and its rows (none, where a short chunk ends before it)
  auto half_row = [](int half) { return REV ? PW_ROWS * (1 - half) : PW_ROWS * half; };
  auto half_rows = [&](const Chunk& k, int half) {
    const int n = k.L - half_row(half);
    // (walking backward it became one vector instruction, and every store a loop over lanes that might differ: 1.68 us a chunk, 1.54 without)
    return (int)fprt::uniform((uint32_t)(n < 0 ? 0 : n < PW_ROWS ? n : PW_ROWS));
  };

  if (wave >= 4) {
    const int fw = wave & 3;
    const uint32_t rowA = (uint32_t)p.H * DA * 2, rowB = (uint32_t)p.H * p.dB * 2;   // bytes between tokens
    const uint32_t headA = (uint32_t)h * DA * 2, headB = ((uint32_t)h * p.dB + (uint32_t)tile * PW_D) * 2;
    Chunk c0 = walk.first(slot), c1 = walk.after(c0);

    // Score tiles: a half's own (on the diagonal) by feed wave 0, that of half 1 with the tokens of half 0 by wave 1
    const bool diagonal = fw == 0;
    float mw[16];
    uint32_t keep[8];      // bits to keep after conversion: a masked score is cleared, so that inf or nan cannot leak through 0 * x
    const int row_at = place(c, g);
    const int p_out = P0 + (diagonal ? 0 : FP_P) + lane * 16;
    auto score_weights = [&]() {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int d = REV ? acc_row(r, g) - c : c - acc_row(r, g);   // distance inside the diagonal tile
        mw[r] = io.s_intra * fprt::exp2_approx((float)(diagonal ? (d >= 0 ? d : 0) : 32 + d) * lg);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int d0 = REV ? acc_row(2 * e, g) - c : c - acc_row(2 * e, g), d1 = REV ? acc_row(2 * e + 1, g) - c : c - acc_row(2 * e + 1, g);
        keep[e] = diagonal ? ((d0 >= 0 ? 0x0000ffffu : 0u) | (d1 >= 0 ? 0xffff0000u : 0u)) : 0xffffffffu;
      }
    };
    u32x4 xf[KS], wf[KS];
    auto score_load = [&](int sx, int sw) {
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        wf[k] = ld128(at((W0 + row_at + sw) ^ (32 * k)));
        xf[k] = ld128(at((X0 + row_at + sx) ^ (32 * k)));
      }
    };
    auto score = [&](int sp) {
      f32x16 sc = {0};
#pragma unroll
      for (int k = 0; k < KS; ++k) sc = fprt::mfma_32x32x16_bf16(wf[k], xf[k], sc);
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        u32x4 d;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int r = 8 * k + 2 * e;
          d[e] = fprt::pack_bf16x2(sc[r] * mw[r], sc[r + 1] * mw[r + 1]) & keep[4 * k + e];
        }
        st128(at(p_out + sp * 2 * FP_P + 1024 * k), d);
      }
    };

    // Y of a half: rows lane / 16 + 4 u, 16 bytes a lane, whole 256-byte pieces of rows.  By wave 0 in the steps of half 0, by wave 1
    // in those of half 1, in which it has no scores to make.
    char* const Yg = reinterpret_cast<char*>(io.Y) + headB;
    const int q_at = Q0 + ((lane & 15) >> 2) * FP_Q + (lane >> 4) * FP_Q_LD + 16 * (lane & 3);
    const uint32_t y_off = (uint32_t)(lane >> 4) * rowB + (lane & 15) * 16;
    auto drain = [&](const Chunk& k, int half, int sp) {
      const int rows = half_rows(k, half);
      const fprt::BufView yv = fprt::make_buf(Yg + (size_t)(k.row + half_row(half)) * rowB, rows > 0 ? (uint32_t)(rows - 1) * rowB + PW_PITCH : 0u);
      u32x4 v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = ld128(at(q_at + sp * 4 * FP_Q + 4 * u * FP_Q_LD));
      // non-temporal: outputs are not read back by this launch and need not displace its inputs in the caches
#pragma unroll
      for (int u = 0; u < 8; ++u) fprt::buf_store128_nt(yv, y_off + 4 * u * rowB, v[u]);
    };
    Chunk cp = c0;
    cp.L = 0;

    if (fw == 0) {
      score_weights();
      fprt::block_sync();
      score_load(0, 0);
      score(0);
      fprt::block_sync();
      int sx = 0, sw = 0;
      auto step = [&](auto half_c, bool last) {
        constexpr int half = decltype(half_c)::value;
        sx = next_x(sx);
        sw = next_w(sw);
        if (!last) score_load(sx, sw);
        if (half == 0) drain(cp, 1, 1);
        if (!last) score(1 - half);
        fprt::block_sync();
      };
#pragma nounroll
      while (true) {
        step(std::integral_constant<int, 0>{}, false);
        step(std::integral_constant<int, 1>{}, c1.L == 0);
        if (c1.L == 0) break;
        cp = c0; c0 = c1;
        c1 = walk.after(c1);
      }
      drain(c0, 1, 1);
      return;
    }

    // ---- copies: of W by wave 1, of X by wave 2, of Z by wave 3.  Copy u: rows 4 u .. + 3 of a tile, whose keys repeat every 16 rows
    const fprt::LdsAddress lds0 = fprt::lds_address(lds);
    const uint32_t pitch = fw == 3 ? rowB : rowA;
    const char* const from = fw == 1 ? reinterpret_cast<const char*>(io.W) + headA : fw == 2 ? reinterpret_cast<const char*>(io.X) + headA
                                                                                           : reinterpret_cast<const char*>(io.Z) + headB;
    const int ring = fw == 1 ? W0 : fw == 2 ? X0 : Z0;
    uint32_t off[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) off[u] = (uint32_t)(4 * u + lane / 16) * pitch + (uint32_t)((lane % 16) ^ key(4 * u + lane / 16)) * 16;
    auto copy = [&](const Chunk& k, int half, int stage) {
      const int rows = half_rows(k, half);
      const fprt::FillView v = fprt::make_fill(from + (size_t)(k.row + half_row(half)) * pitch, rows > 0 ? (uint32_t)(rows - 1) * pitch + PW_PITCH : 0u);
      uint32_t offs[COPIES];
#pragma unroll
      for (int u = 0; u < COPIES; ++u) offs[u] = off[u & 3] + (u >> 2) * 16 * pitch;
      fprt::fill_lds<false, 1024>(v, offs, lds0 + (ring + stage));
    };
    // W weighted for the state update, by waves 2 and 3: rows 4 u + lane / 16, u = 4 (fw - 2) .. + 3
    auto weight = [&](int half, int u, int L) {
      const int j = half_row(half) + 4 * u + lane / 16;
      int e = REV ? j + 1 : L - 1 - j;
      if (e < 0) e = 0;   // rows beyond a short chunk are zeros, their weight only has to be finite
      return io.s_update * fprt::exp2_approx((float)e * lg);
    };
    float w_full[2][4];
    auto weigh = [&](const Chunk& k, auto half_c, int sw, int sp) {
      constexpr int half = decltype(half_c)::value;
      u32x4 v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = ld128(at(W0 + sw + 1024 * (4 * (fw & 1) + i) + 16 * lane));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int u = 4 * (fw & 1) + i;
        const float w = REV || k.L == CH ? w_full[half][i] : weight(half, u, k.L);
        u32x4 o;
#pragma unroll
        for (int d = 0; d < 4; ++d) o[d] = fprt::pack_bf16x2(bf16_elem(v[i], 2 * d) * w, bf16_elem(v[i], 2 * d + 1) * w);
        st128(at(WW0 + sp * PW_TILE + 1024 * u + 16 * lane), o);
      }
    };
    // Chunks j, j + 1, j + 2; steps 2 j and 2 j + 1 carry chunk j.  Chunks that do not exist are copied through empty views, so that
    // the counts hold.
    Chunk c2 = walk.after(c1);
    copy(c0, 0, 0);
    copy(c0, 1, PW_TILE);
    copy(c1, 0, 2 * PW_TILE);
    copy(c1, 1, 3 * PW_TILE);
    if (fw == 1) {
      score_weights();
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) w_full[i >> 2][i & 3] = weight(i >> 2, 4 * (fw & 1) + (i & 3), CH);
    }
    fprt::fill_wait<3 * COPIES>();
    fprt::block_sync();
    if (fw >= 2) weigh(c0, std::integral_constant<int, 0>{}, 0, 0);
    fprt::fill_wait<2 * COPIES>();
    fprt::block_sync();
    int sx = 0, sw = 0;   // stages of the step's half
    bool first = true;
    // Step `half` of chunk c0: half `half` of chunk c2 is asked for, the half after the step's weighed or scored.  That one has
    // arrived, and before the step ends the next: asked for two steps ago, with two halves' copies after it.
    auto step = [&](auto half_c, bool last) {
      constexpr int half = decltype(half_c)::value;
      constexpr int nh = 1 - half;
      const int sx1 = next_x(sx), sw1 = next_w(sw), sw4 = sw == 0 ? AHEAD * PW_TILE : sw - PW_TILE;
      if (fw == 1) {
        if (nh == 1) score_load(sx1, sw);
        else drain(c0, 0, 0);
      }
      copy(c2, half, fw == 2 ? sx : sw4);
      if (fw == 1) {
        if (nh == 1) score(nh);
      } else if (!last) {
        weigh(half == 0 ? c0 : c1, std::integral_constant<int, nh>{}, sw1, nh);
      }
      // (wave 1: and a half's outputs, but in the first step)
      if (fw == 1 && !(half == 0 && first)) fprt::fill_wait<2 * COPIES + 8>();
      else fprt::fill_wait<2 * COPIES>();
      first = false;
      fprt::block_sync();
      sx = sx1;
      sw = sw1;
    };
#pragma nounroll
    while (true) {
      step(std::integral_constant<int, 0>{}, false);
      step(std::integral_constant<int, 1>{}, c1.L == 0);
      if (c1.L == 0) break;
      c0 = c1; c1 = c2;
      c2 = walk.after(c2);
    }
    fprt::fill_wait<0>();   // (nothing may arrive after the end)
    return;
  }

  // ================================= carry waves =================================
  const int ns = wave;                          // this wave: columns 32 ns ..
  // racc[a] element r is R[32 a + 16 (r / 8) + 8 g + r % 8][n], n = 32 ns + swapped(c)
  f32x16 racc[NAB];
#pragma unroll
  for (int a = 0; a < NAB; ++a) racc[a] = f32x16{0};

  // ---- R <-> a state matrix in global memory, 16 bytes per lane along the contiguous direction of the matrix.  R = S^T (`tposed`): the
  // pieces are this lane's elements.  R = S: a block of 32 rows at a time, turned in this wave's quarter of output stage 0, which is not in use.
  const bool tposed = io.rs_a == 1;
  const uint32_t mat_bytes = (uint32_t)p.dA * (uint32_t)p.dB * 2;
  auto matrix = [&](auto* base) { return base + ((size_t)slot * p.H + h) * p.dA * p.dB; };
  const uint32_t m_step = 2u * (tposed ? 16u : 16u * (uint32_t)io.rs_a);   // from one group of 16 rows to the next
  auto m_offset = [&]() {
    const int l = fprt::opaque(lane);
    return 2u * (tposed ? (uint32_t)((tile * PW_D + 32 * ns + swapped(l & 31)) * (int)io.rs_n + 8 * (l >> 5))
                        : (uint32_t)((l >> 2) * (int)io.rs_a + tile * PW_D + 32 * ns + 8 * (l & 3)));
  };
  const int quarter = Q0 + ns * FP_Q;
  auto turn_offset = [&]() {
    const int l = fprt::opaque(lane);
    return quarter + (l >> 2) * FP_Q_LD + 16 * (l & 3);
  };
  // elements 8 (i % 2) .. + 7 of racc[i / 2], i = 0 .. 2 NAB - 1, in d
  auto load_strip = [&](u32x4 (&d)[2 * NAB], const uint16_t* src) {
    const fprt::BufView view = fprt::make_buf(src, mat_bytes);
    const uint32_t off = m_offset();
#pragma unroll
    for (int i = 0; i < 2 * NAB; ++i) d[i] = fprt::buf_load128(view, off + i * m_step);
    if (tposed) return;
    const int l = fprt::opaque(lane), to = turn_offset();
    const int from = quarter + (8 * (l >> 5) + ((l & 15) >> 2)) * FP_Q_LD + 32 * ((l >> 4) & 1) + 8 * swap2(l & 3);
#pragma unroll
    for (int a = 0; a < NAB; ++a) {
      st128(at(to), d[2 * a]);
      st128(at(to + 16 * FP_Q_LD), d[2 * a + 1]);
      fprt::wave_sync();
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
        d[2 * a + hf] = joined(fprt::lds_read_tr16_b64(at(from + 16 * hf * FP_Q_LD)), fprt::lds_read_tr16_b64(at(from + (16 * hf + 4) * FP_Q_LD)));
      fprt::wave_sync();
    }
  };
  Chunk cur = walk.first(slot), nxt = walk.after(cur);
  if (io.R0) {
    u32x4 upper[2 * NAB], lower[2 * NAB];
    load_strip(upper, matrix(io.R0));
    if (io.R0lo) load_strip(lower, matrix(io.R0lo));
#pragma unroll
    for (int i = 0; i < 2 * NAB; ++i) {
#pragma unroll
      for (int e = 0; e < 8; ++e) racc[i >> 1][8 * (i & 1) + e] = io.R0lo ? joined_elem(upper[i], lower[i], e) : bf16_elem(upper[i], e);
    }
  }
  // Operands read along the tokens: tokens 16 k + 4 g + {0..3} and + 8 of k-step k, columns in `swapped` order
  const int tr_row = 4 * g + ((lane & 15) >> 2), tr_piece = 2 * ((lane >> 4) & 1) + (swap2(lane & 3) >> 1), tr_in = 8 * (swap2(lane & 3) & 1);
  const int z_lo = Z0 + place(tr_row, 4 * ns + tr_piece) + tr_in, z_hi = Z0 + place(tr_row + 8, 4 * ns + tr_piece) + tr_in;
  const int w_lo = WW0 + place(tr_row, tr_piece) + tr_in, w_hi = WW0 + place(tr_row + 8, tr_piece) + tr_in;   // ^ 64 a: columns 32 a ..
  const int x_at = X0 + place(c, g);
  // read-out weights of a full chunk's halves
  const int i0 = half_row(0) + c, i1 = half_row(1) + c;
  const float wread_full0 = io.s_read * fprt::exp2_approx((float)(REV ? CH - 1 - i0 : i0 + 1) * lg);
  const float wread_full1 = io.s_read * fprt::exp2_approx((float)(REV ? CH - 1 - i1 : i1 + 1) * lg);
  const float gL_full = fprt::exp2_approx((float)CH * lg);
  const int p_at = P0 + lane * 16;
  const int y_at = quarter + c * FP_Q_LD + 16 * g;

  fprt::block_sync();
  u32x4 xf[KS], ra[KS], zp[2];   // ra: the R that the chunk starts with; zp: half 0's rows of Z
  int sx = 0, sw = 0;
#pragma unroll
  for (int k = 0; k < KS; ++k) xf[k] = ld128(at(x_at ^ (32 * k)));
  fprt::block_sync();

  auto step = [&](auto half_c, int L) {
    constexpr int half = decltype(half_c)::value;
    u32x4 z[2], pd[2], po[2], wa[2][NAB];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      z[k] = joined(fprt::lds_read_tr16_b64(at(z_lo + sw + 16 * k * PW_PITCH)), fprt::lds_read_tr16_b64(at(z_hi + sw + 16 * k * PW_PITCH)));
      pd[k] = ld128(at(p_at + half * 2 * FP_P + 1024 * k));
      if (half == 1) po[k] = ld128(at(p_at + half * 2 * FP_P + FP_P + 1024 * k));
    }
    // ---- read-out of the R that the chunk starts with, Y^T[n][i] = sum_a R[a][n] X[i][a]
    f32x16 acc = {0};
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      if (half == 0) ra[k] = packed(racc[k >> 1], k & 1);
      acc = fprt::mfma_32x32x16_bf16(ra[k], xf[k], acc);
    }
    fprt::sched_fence();
    auto request_w = [&](int k) {
#pragma unroll
      for (int a = 0; a < NAB; ++a)
        wa[k][a] = joined(fprt::lds_read_tr16_b64(at(((w_lo + half * PW_TILE) ^ (64 * a)) + 16 * k * PW_PITCH)),
                          fprt::lds_read_tr16_b64(at(((w_hi + half * PW_TILE) ^ (64 * a)) + 16 * k * PW_PITCH)));
    };
    request_w(0);
    sx = next_x(sx);
#pragma unroll
    for (int k = 0; k < KS; ++k) xf[k] = ld128(at((x_at + sx) ^ (32 * k)));
    float wread = half == 0 ? wread_full0 : wread_full1;
    if (REV && L != CH) {
      const int i = half == 0 ? i0 : i1;
      wread = io.s_read * fprt::exp2_approx((float)(i < L ? L - 1 - i : 0) * lg);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] *= wread;
    if (half == 0) {
      float gL = gL_full;
      if (L != CH) gL = fprt::exp2_approx((float)L * lg);
#pragma unroll
      for (int a = 0; a < NAB; ++a) {
#pragma unroll
        for (int r = 0; r < 16; ++r) racc[a][r] *= gL;
      }
    }
    // The two tiles of half 1 are summed in the order of retention_pass_ws.h, whose waves begin with the tile that they made themselves,
    // those of the odd column blocks the other one: a call's o has the same bits whether it leaves block states (there) or not (here)
    auto own_tile = [&]() {
#pragma unroll
      for (int k = 0; k < 2; ++k) acc = fprt::mfma_32x32x16_bf16(z[k], pd[k], acc);
    };
    auto other_tile = [&]() {
#pragma unroll
      for (int k = 0; k < 2; ++k) acc = fprt::mfma_32x32x16_bf16(zp[k], po[k], acc);
    };
    if (half == 0) {
      own_tile();
    } else if (ns & 1) {
      other_tile();
      own_tile();
    } else {
      own_tile();
      other_tile();
    }
    fprt::sched_fence();
    request_w(1);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
#pragma unroll
      for (int a = 0; a < NAB; ++a) racc[a] = fprt::mfma_32x32x16_bf16(wa[k][a], z[k], racc[a]);
      if (half == 0) zp[k] = z[k];
    }
    // accumulator element r of Y^T is column 16 (r / 8) + 8 g + r % 8 of this wave's quarter
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) st128(at(y_at + half * 4 * FP_Q + 32 * hf), packed(acc, hf));
    fprt::block_sync();
    sw = next_w(sw);
  };
#pragma nounroll
  while (true) {
    step(std::integral_constant<int, 0>{}, cur.L);
    step(std::integral_constant<int, 1>{}, cur.L);
    if (nxt.L == 0) break;
    cur = nxt;
    nxt = walk.after(nxt);
  }
  if (io.Rout) {   // (output stage 0: drained)
    const fprt::BufView view = fprt::make_buf(matrix(io.Rout), mat_bytes);
    const uint32_t off = m_offset();
    const int l = fprt::opaque(lane), from = turn_offset();
#pragma unroll
    for (int a = 0; a < NAB; ++a) {
      if (tposed) {
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) fprt::buf_store128(view, off + (2 * a + hf) * m_step, packed(racc[a], hf));
        continue;
      }
#pragma unroll
      for (int r = 0; r < 16; ++r)
        reinterpret_cast<u16_m*>(at(quarter + (16 * (r >> 3) + 8 * (l >> 5) + (r & 7)) * FP_Q_LD))[swapped(l & 31)] = float_to_bf16_bits(racc[a][r]);
      fprt::wave_sync();
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) fprt::buf_store128(view, off + (2 * a + hf) * m_step, ld128(at(from + 16 * hf * FP_Q_LD)));
      fprt::wave_sync();
    }
  }
}

FP_DEVICE void retention_pass_wide(const PassArgs& p, const PassTensors& io, char* lds, int wg) {
  if (io.reverse) retention_pass_wide_dir<true>(p, io, lds, wg);
  else retention_pass_wide_dir<false>(p, io, lds, wg);
}

// Whether a launch of `passes` planned plain passes takes this kernel: where workgroups of 64 columns would not fit the device at once,
// and, where these do not either, of sequences that are worth a workgroup (the others go from sequence to sequence with the next one's
// rows on their way).  Speed over the pass kernel's, which it has for dA = 128 otherwise, forward / backward, 256 units, by workgroups here:
//                   144 (128 x 128: 160)      256                       528 (264 at 128 x 256)    1024 (512)
//   128 x 128  T64     1.36 / 1.29            1.16 / 1.11               .84 / .81                 .90 / .89
//              T256    1.44 / 1.35            1.26 / 1.22               .98 / .98                 .96 / 1.01
//              T512    1.52 / 1.45            1.26 / 1.25               1.01 / 1.02               1.07 / 1.07
//              T2048   1.41 / 1.41            1.13 / 1.14               1.17 / 1.16 (512)         1.16 / 1.16 (768)
//   128 x 256  T64     1.32 / 1.24            1.28 / 1.20               .88 / .83                 .99 / .94
//              T128    1.41 / 1.32            1.25 / 1.19               1.03 / .96                1.08 / 1.04
//              T192    1.46 / 1.38            1.34 / 1.26               1.10 / 1.06               1.16 / 1.16
//              T2048   1.71 / 1.66            1.46 / 1.38               1.33 / 1.28               1.45 / 1.39 (512)
// Where 64 columns each fill half of the device or less, a step there is as long as one here and there are twice as many (128 x 128,
// 64 to 256 of them: .87 to .96; 128 x 256, 256 of them: 1.00 to 1.03).
inline bool pass_is_wide(const PassArgs& a, int passes, int compute_units) {
  if (a.dA != PW_D || a.dB % PW_D != 0) return false;
  const long long wgs = (long long)passes * a.B * a.H * (a.dB / PW_D);
  return 2 * wgs > compute_units && (wgs <= compute_units || (long long)a.T * a.dB >= 384 * 128);
}

}  // namespace fpk
