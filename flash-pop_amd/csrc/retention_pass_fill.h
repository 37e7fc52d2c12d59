// Retention pass (see pass_args.h for the recurrence) whose tiles go from global memory into LDS without passing through
// registers: dA = 64; of the walks with suffixes the forward one whose suffixes fit beside a chunk.
//
// One workgroup owns one (batch, head) stream and 64 columns of Z, Y and R.  Its waves have one of three roles:
//
//   carry  (4 waves)  each a strip of 32 columns of R in fp32 accumulators and 32 of a chunk's rows (two waves hold the same
//                     strip).  The rows of a converted accumulator tile are put in such an order (`swapped`) that it is the
//                     read-out's operand as it is: R never goes through LDS.  Read-out, product with Z, output, state update.
//   score  (4 waves)  one chunk ahead of them, the score tiles; the way out of the chunk before
//   move   (4 waves)  the copies of later chunks into LDS, W of the next chunk weighted for the state update
//
// One workgroup barrier per chunk: what a wave reads between two barriers was written before the first of them.
//
//   step i   copied into LDS  chunk i + AHEAD     scores, weighted W, X fragments  i + 1
//            carried          chunk i             on its way out                   i - 1
//
// The tiles are row-major; the 16-byte pieces of a row are exchanged by a XOR with a key of the row (FillTile), which a copy
// does by the global address that a lane reads from.  Both 16 consecutive rows at one piece (row-wise operands) and four
// consecutive rows at four neighbouring pieces (a transposing read's 32 lanes) are then on different banks, without padding.
//
// What bounds it: on a few workgroups the carry waves' chain (0.67 us of a step's 0.78; one chunk from start to end 4.0 us, launches in a
// row), on many the memory.  Three roles of 12 waves against two of 8, whose feed waves were as long a chain as the carry waves: 0.94 us
// a step.  The walk of retention_pass_ws.h (rows through registers, tiles transposed on the way, scores and product with Z in one
// chunk's time behind a second barrier), which this replaces for dA = 64, against it here, us a launch, launches in a row:
//   64 x 64    4 workgroups     T64 4.42 -> 4.03   T256 7.70 -> 6.3    T512 11.9 -> 9.2    T4096 71.9 -> 50.4
//              128 (H4)         T64 4.90 -> 4.5    T256 8.5 -> 7.6     T2048 41.6 -> 34.1
//              256 (H4)         T64 5.3 -> 4.8     T256 9.5 -> 8.8     T2048 52.0 -> 50.8
//   64 x 128   96 (B4 H12)      T64 4.8 -> 4.4     T256 8.3 -> 7.2     T2048 38.4 -> 30.6
//              240 (B10 H12)    T64 5.2 -> 4.8     T256 9.1 -> 8.1     T2048 45.9 -> 41.7
// The same for dA = 128 was slower from 96 workgroups on (128: 50 -> 56 us): LDS holds the rows of one chunk less ahead.
#pragma once
#include "pass_args.h"
#include "lds_access.h"

namespace fpk {

constexpr int FP_DA = 64;                 // columns of X and W
constexpr int FP_THREADS = 768;
constexpr int FP_AHEAD = 3;               // chunks between the step that asks for a chunk's rows and the one that carries it
constexpr int FP_P = 2 * 32 * 32;         // bytes of a score tile: [k-step][lane][8]
constexpr int FP_Q_LD = 2 * (32 + 8);     // row pitch of a carry wave's quarter of the staged output, bytes
constexpr int FP_Q = 32 * FP_Q_LD;

// FILL_MULTI: a workgroup may walk several sequences (p.slots < p.B); FILL_BLOCKS: chunks end at block boundaries, where block
// states leave (Bout, walking forward) or their gradients join (Bin, walking backward).  FILL_FOLD: chunks end at block boundaries
// of a POP call, and a suffix of at most FP_SFX tokens is part of the chunk that starts at its boundary, whose state it reads: a
// fourth score tile, a second read-out, 16 more rows of every tensor.  The suffix at T hangs off one more, empty, chunk.
enum FillMode { FILL_PLAIN = 0, FILL_MULTI = 1, FILL_BLOCKS = 2, FILL_FOLD = 3 };
constexpr int FP_SFX = 16;

// A tile of 64 tokens x 64 features
struct FillTile {
  static constexpr int PITCH = 2 * 64;           // bytes
  static constexpr int BYTES = CH * PITCH;
  static constexpr int PPR = 8;                  // 16-byte pieces per row
  static constexpr int ROWS = 64 / PPR;          // rows that one copy of a wave covers
  static constexpr int PER_WAVE = CH / ROWS / 4; // copies of each of four waves
  static FP_DEVICE int key(int row) { return (((row >> 1) & 1) << 2) | ((row >> 2) & 3); }
  // byte offset of piece p of a row
  static FP_DEVICE int at(int row, int p) { return row * PITCH + 16 * (p ^ key(row)); }
};
static_assert(FP_DA == 64 && BV == 64, "one tile shape for X, W and Z");
constexpr int fp_lds_bytes() {
  return FP_AHEAD * 2 * FillTile::BYTES       // X, W
         + (FP_AHEAD + 1) * FillTile::BYTES   // Z
         + 2 * FillTile::BYTES                // W weighted
         + 2 * 3 * FP_P                       // scores
         + 2 * 4 * FP_Q                       // staged output
         + 4 * FillTile::BYTES;               // states that enter; FILL_FOLD: the suffixes' tiles
}

namespace pp {

// Accumulator row / operand row m of a group of 16 stands for position 8 (bit 2) + 4 (bit 3) + (bits 0, 1): a lane then holds
// eight consecutive positions per k-step.
FP_DEVICE int swap2(int q) { return ((q & 1) << 1) | ((q >> 1) & 1); }
FP_DEVICE int swapped(int m) { return (m & ~12) | (swap2((m >> 2) & 3) << 2); }
FP_DEVICE u32x4 packed(const f32x16& v, int half) {
  u32x4 d;
#pragma unroll
  for (int e = 0; e < 4; ++e) d[e] = fprt::pack_bf16x2(v[8 * half + 2 * e], v[8 * half + 2 * e + 1]);
  return d;
}
FP_DEVICE u32x4 joined(u32x2 lo, u32x2 hi) { return u32x4{lo[0], lo[1], hi[0], hi[1]}; }

// A chunk of a walk: the next `L` (0: beyond the walk) of the `left` tokens that its sequence still has in walking order
struct Chunk {
  int L, left;
  uint32_t row;        // its first row among all rows of a tensor
  int b;               // its sequence
  bool first;          // starts its sequence
  int bound, blk;      // FILL_BLOCKS, FILL_FOLD: tokens up to the next boundary, block that the chunk belongs to
  int sfx;             // FILL_FOLD: the suffix at its first token, -1: none
  uint32_t base;       // the sequence's first row
  int len;             // ... and tokens
};
FP_DEVICE bool live(const Chunk& k) { return k.L > 0 || k.sfx >= 0; }
// The chunks of sequence `slot`, then (FILL_MULTI) of slot + slots, ...  Without divisions and, but for a change of the sequence, branches.
template <int MODE, bool REV>
struct ChunkWalk {
  const PassArgs& p;
  FP_DEVICE void place(Chunk& k) const {
    k.L = k.left < CH ? k.left : CH;
    if (MODE == FILL_BLOCKS || MODE == FILL_FOLD) k.L = k.bound < k.L ? k.bound : k.L;
    k.row = REV ? k.base + (uint32_t)(k.left - k.L) : k.base + (uint32_t)(k.len - k.left);
  }
  FP_DEVICE Chunk first(int b) const {
    Chunk k;
    k.b = b;
    k.first = true;
    k.len = p.T;
    k.base = (uint32_t)b * p.T;
    if ((MODE == FILL_PLAIN || MODE == FILL_MULTI) && p.segs > 0) {   // (the last segment may be shorter)
      const int seg = b % p.segs, left = p.total - seg * p.T;
      k.len = left < p.T ? left : p.T;
      k.base = (uint32_t)(b / p.segs) * p.total + (uint32_t)seg * p.T;
    }
    k.left = b < p.B ? k.len : 0;
    k.blk = k.bound = 0;
    k.sfx = MODE == FILL_FOLD ? 0 : -1;
    if (MODE == FILL_BLOCKS || MODE == FILL_FOLD) {
      k.blk = REV ? (p.T - 1) / p.block : 0;
      k.bound = REV ? p.T - k.blk * p.block : p.block;
    }
    place(k);
    return k;
  }
  FP_DEVICE Chunk after(const Chunk& k) const {
    Chunk n = k;
    n.left = k.left - k.L;
    n.first = false;
    if (MODE == FILL_MULTI && k.L > 0 && n.left == 0) return first(k.b + p.slots);
    if (MODE == FILL_BLOCKS || MODE == FILL_FOLD) {
      const bool crosses = k.bound == k.L;
      n.bound = crosses ? p.block : k.bound - k.L;
      n.blk = k.blk + (crosses ? (REV ? -1 : 1) : 0);
      if (MODE == FILL_FOLD) n.sfx = crosses && k.L > 0 ? n.blk : -1;
    }
    place(n);
    return n;
  }
  // whether the state after a chunk (before it, walking backward) is that behind a full block, block k.blk
  FP_DEVICE bool at_block_end(const Chunk& k) const {
    if (MODE != FILL_BLOCKS || k.L == 0) return false;
    return REV ? k.bound == p.block && (k.blk + 1) * p.block <= p.T : k.bound == k.L;
  }
};

}  // namespace pp

// Whether a pass moves more than the caches hold; rows of such a one that nobody reads again are copied with the cache hint (below, the
// next launch finds some of them: the backward behind the forward of B32 T2048 H4 64 x 64, 134 MB, 60 us, 65 with the hint in the
// forward).  Forward alone, and forward and backward of a training step, cold inputs, us: this rule; no hint at all; the hint on every row
// of every launch:
//   64 x 64    B64 T2048 H4     53.4, 170.7     56.2, 174.4     53.3, 181.1
//              B64 T4096 H4     101.8, 344.7    108.3, 352.5    102.2, 365.5
//   64 x 128   B16 T2048 H12    67.4, 223.2     70.7, 227.3     77.7, 235.2
//              B32 T2048 H12    123.9, 419.4    141.1, 425.2    161.2, 429.2
//   64 x 256   B16 T2048 H8     71.3, 259.0     77.3, 263.1     74.7, 266.6
FP_DEVICE bool passes_caches(const PassArgs& p) { return (size_t)p.B * p.T * p.H * (p.dA + p.dB) * 4 > (200u << 20); }

// Workgroup number `wg` of a pass; `io`: the tensors, walking direction and scales of this pass (a launch may hold several,
// everything else in `p` is common to them).  ALONE: the launch holds this pass only.
template <int MODE, bool REV, bool ALONE>
FP_DEVICE void retention_pass_fill_dir(const PassArgs& p, const PassTensors& io, char* lds, int wg) {
  using namespace pp;
  using TT = FillTile;
  constexpr bool MULTI = MODE == FILL_MULTI, BLOCKS = MODE == FILL_BLOCKS, FOLD = MODE == FILL_FOLD;
  static_assert(!FOLD || !REV, "suffixes: forward only");
  constexpr int DA = FP_DA, AHEAD = FP_AHEAD, KS = DA / 16, NAB = DA / 32;
  constexpr int COPIES = 3 * TT::PER_WAVE + (FOLD ? 2 : 0);   // of a move wave, per chunk
  static_assert(AHEAD == 3, "the waits below");

  // X and W of a chunk are done with when it is carried, Z a step later
  constexpr int X0 = 0, W0 = X0 + AHEAD * TT::BYTES, Z0 = W0 + AHEAD * TT::BYTES, WW0 = Z0 + (AHEAD + 1) * TT::BYTES,
                P0 = WW0 + 2 * TT::BYTES, Q0 = P0 + 2 * 3 * FP_P,
                END = Q0 + 2 * 4 * FP_Q, S0 = FOLD ? Q0 : END;
  // FOLD: tiles of 16 rows (X and Z are both read when the chunk is carried); the state that enters takes the output stages' place
  constexpr int SB = FP_SFX * TT::PITCH, XS0 = END, WS0 = XS0 + (AHEAD + 1) * SB, ZS0 = WS0 + AHEAD * SB, PS0 = ZS0 + (AHEAD + 1) * SB,
                QS0 = PS0 + 2 * FP_P / 2, QS_HALF = FP_SFX * FP_Q_LD, QS_STAGE = 2 * QS_HALF;
  static_assert(QS0 + 2 * QS_STAGE <= fp_lds_bytes() && S0 + 4 * TT::BYTES * (FOLD ? 0 : 1) <= fp_lds_bytes() && TT::BYTES <= 2 * 4 * FP_Q, "the tiles fit");
  auto at = [&](int byte) { return reinterpret_cast<uint16_t*>(lds + byte); };
  // the stage after one that starts `off` bytes into the rings of X and W, into that of Z
  auto next_x = [](int off) { return off == (AHEAD - 1) * TT::BYTES ? 0 : off + TT::BYTES; };
  auto next_z = [](int off) { return off == AHEAD * TT::BYTES ? 0 : off + TT::BYTES; };

  const int tid = fprt::thread_index(), wave = (int)fprt::uniform((uint32_t)tid >> 6), lane = tid & 63, g = lane >> 5, c = lane & 31;
  const int ntile = p.dB / BV;
  const int tile = wg % ntile, h = (wg / ntile) % p.H, slot = (wg / ntile) / p.H;
  const float lg = p.log2g[h];
  const ChunkWalk<MODE, REV> walk{p};

  // A chunk that starts with a state of its own: an initial one (MULTI), or a block state's gradient that joins (BLOCKS walking
  // backward).  These and the first are copied into LDS like the rows, this workgroup's 64 columns of R, [a][n] or, where R = S^T
  // (`tposed`), [n][a].  Four tiles taken in turn, or two pairs where the states are fp32, upper and lower halves.
  const bool tposed = io.rs_a == 1, halves = io.R0lo != nullptr;
  auto sfx_row = [&](const Chunk& k) { return ((uint32_t)k.b * (p.nblk + 1) + (k.sfx > 0 ? k.sfx : 0)) * p.Ls; };
  auto brings_state = [&](const Chunk& k) { return MULTI ? io.R0 && k.first && k.L > 0 : BLOCKS && REV && io.Bin && walk.at_block_end(k); };
  auto state_tile = [&](int n) { return S0 + (halves ? (n & 1) * 2 : n & 3) * TT::BYTES; };
  auto matrix = [&](auto* base, int b) { return base + ((size_t)b * p.H + h) * p.dA * p.dB; };
  auto block_matrix = [&](auto* base, const Chunk& k) { return matrix(base, k.b * p.nblk + k.blk); };

  const uint32_t rowA = (uint32_t)p.H * DA * 2, rowB = (uint32_t)p.H * p.dB * 2;   // bytes between tokens
  const uint32_t headA = (uint32_t)h * DA * 2, headB = ((uint32_t)h * p.dB + (uint32_t)tile * BV) * 2;

  if (wave >= 8) {
    // ================================= move waves =================================
    const int fw = wave & 3;
    // Copy u of this wave: rows ROWS (fw + 4 u) .. of a tile, whose keys do not depend on u
    const int row0 = TT::ROWS * fw + lane / TT::PPR, piece = (lane % TT::PPR) ^ TT::key(row0);
    const uint32_t offA = (uint32_t)row0 * rowA + (uint32_t)piece * 16, offB = (uint32_t)row0 * rowB + (uint32_t)piece * 16;
    const fprt::LdsAddress lds0 = fprt::lds_address(lds);
    const char* const Xg = reinterpret_cast<const char*>(io.X) + headA;
    const char* const Wg = reinterpret_cast<const char*>(io.W) + headA;
    const char* const Zg = reinterpret_cast<const char*>(io.Z) + headB;
    // X and W with the hint only where no other column tile reads them, nothing where several passes of a launch read the same rows.  A
    // forward that leaves block states (checkpoints) has a backward behind it, which starts where it ended and reads q once but k and v twice:
    // there X alone.
    const bool once = ALONE && passes_caches(p), x_once = once && ntile == 1, w_once = x_once && !BLOCKS, z_once = once && !BLOCKS;
    // this wave's part of 64 rows into a tile at `to`
    auto fill = [&](const fprt::FillView& v, uint32_t off, uint32_t pitch, int to, bool hint) {
      const fprt::LdsAddress dst = lds0 + (to + 1024 * fw);
      const uint32_t offs[TT::PER_WAVE] = {off, off + 4 * TT::ROWS * pitch};
      if (hint) fprt::fill_lds<true, 4096>(v, offs, dst);
      else fprt::fill_lds<false, 4096>(v, offs, dst);
    };
    auto copy_w = [&](const Chunk& k, int sx) {
      fill(fprt::make_fill(Wg + (size_t)k.row * rowA, k.L > 0 ? (uint32_t)(k.L - 1) * rowA + DA * 2 : 0u), offA, rowA, W0 + sx, w_once);
    };
    auto copy_xz = [&](const Chunk& k, int sx, int sz) {
      fill(fprt::make_fill(Xg + (size_t)k.row * rowA, k.L > 0 ? (uint32_t)(k.L - 1) * rowA + DA * 2 : 0u), offA, rowA, X0 + sx, x_once);
      fill(fprt::make_fill(Zg + (size_t)k.row * rowB, k.L > 0 ? (uint32_t)(k.L - 1) * rowB + BV * 2 : 0u), offB, rowB, Z0 + sz, z_once);
    };
    // FOLD: the 16 rows of a tensor are two copies, of X by wave 0, of W by wave 1 and of Z by the other two (as many each)
    auto copy_suffix = [&](const Chunk& k, int sx, int sz) {
      if constexpr (FOLD) {
        const uint32_t pitch = fw < 2 ? rowA : rowB;
        const char* const from = (fw == 0 ? reinterpret_cast<const char*>(io.Xs) + headA : fw == 1 ? reinterpret_cast<const char*>(io.Ws) + headA
                                                                                               : reinterpret_cast<const char*>(io.Zs) + headB);
        const int to = fw == 0 ? XS0 + sz / (TT::BYTES / SB) : fw == 1 ? WS0 + sx / (TT::BYTES / SB) : ZS0 + sz / (TT::BYTES / SB);
        const fprt::FillView v = fprt::make_fill(from + (size_t)sfx_row(k) * pitch, k.sfx >= 0 ? (uint32_t)(p.Ls - 1) * pitch + 128 : 0u);
        uint32_t off[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int row = TT::ROWS * u + lane / TT::PPR;
          off[u] = (uint32_t)row * pitch + (uint32_t)((lane % TT::PPR) ^ TT::key(row)) * 16;
        }
        fprt::fill_lds<false, 1024>(v, off, lds0 + to);
      }
    };
    auto copy = [&](const Chunk& k, int sx, int sz) {
      copy_w(k, sx);
      copy_xz(k, sx, sz);
      copy_suffix(k, sx, sz);
    };
    const uint32_t rowR = 2u * (uint32_t)(tposed ? io.rs_n : io.rs_a);
    auto copy_tile = [&](const uint16_t* m, int to) {
      const fprt::FillView v = fprt::make_fill(reinterpret_cast<const char*>(m) + (tposed ? (size_t)tile * BV * rowR : (size_t)tile * BV * 2), 63 * rowR + 128);
      const int l = fprt::opaque(lane);
      const uint32_t off = (uint32_t)(TT::ROWS * fw + l / TT::PPR) * rowR + (uint32_t)((l % TT::PPR) ^ TT::key(row0)) * 16;
      fill(v, off, rowR, to, false);
    };
    int states = 0;   // asked for so far
    auto copy_initial = [&](int b) {
      copy_tile(matrix(io.R0, b), state_tile(states));
      if (halves) copy_tile(matrix(io.R0lo, b), state_tile(states) + TT::BYTES);
      ++states;
    };
    auto copy_state = [&](const Chunk& k) {
      if (MULTI) {
        copy_initial(k.b);
      } else {
        copy_tile(block_matrix(io.Bin, k), state_tile(states));
        ++states;
      }
    };
    // Rows 8 u + lane / 8 of W, u = fw and fw + 4, weighted for the state update, in the places that they have in their tile
    auto weight = [&](int u, int L) {
      const int j = 8 * u + (lane >> 3);
      int e = REV ? j + 1 : L - 1 - j;
      if (e < 0) e = 0;   // rows beyond a short chunk are zeros, their weight only has to be finite
      return io.s_update * fprt::exp2_approx((float)e * lg);
    };
    const float w_full[2] = {weight(fw, CH), weight(fw + 4, CH)};
    auto weigh = [&](const Chunk& k, int sx, int sp) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int u = fw + 4 * i;
        const float w = REV || k.L == CH ? w_full[i] : weight(u, k.L);
        const u32x4 v = ld128(at(W0 + sx + 1024 * u + 16 * lane));
        u32x4 o;
#pragma unroll
        for (int d = 0; d < 4; ++d) o[d] = fprt::pack_bf16x2(bf16_elem(v, 2 * d) * w, bf16_elem(v, 2 * d + 1) * w);
        st128(at(WW0 + sp * TT::BYTES + 1024 * u + 16 * lane), o);
      }
    };

    // chunks i, ..., i + AHEAD; those that do not exist are copied through empty views, so that the counts hold
    Chunk c0 = walk.first(slot), c1 = walk.after(c0), c2 = walk.after(c1), c3 = walk.after(c2);
    if (io.R0) copy_initial(c0.b);
    if (!MULTI && brings_state(c0)) copy_state(c0);
    copy(c0, 0, 0);
    if (brings_state(c1)) copy_state(c1);
    copy(c1, TT::BYTES, TT::BYTES);
    copy(c2, 2 * TT::BYTES, 2 * TT::BYTES);
    fprt::fill_wait<2 * COPIES>();
    fprt::block_sync();
    weigh(c0, 0, 0);
    fprt::fill_wait<COPIES>();
    fprt::block_sync();
    int sx = 0, sz = 0, sp = 0;   // stages of chunk i
    bool late = false;            // the state of chunk i + 1 has not been asked for
#pragma nounroll
    while (live(c1)) {
      // The rows of W and those of X and Z not at once: where T * H * dA is a power of two all of them are on the same channels of
      // the memory (B16 T4096 H16, 64 values: 112 -> 101 us a launch).
      const int sx1 = next_x(sx);
      if (late) copy_state(c1);
      // two pairs: the third state in a row has to wait until the first was taken
      const bool due = brings_state(c2);
      late = due && halves && brings_state(c0) && brings_state(c1);
      const bool state = due && !late;
      if (state) copy_state(c2);
      copy_w(c3, sx);
      weigh(c1, sx1, sp ^ 1);
      const int sz3 = sz == 0 ? AHEAD * TT::BYTES : sz - TT::BYTES;
      copy_xz(c3, sx, sz3);
      copy_suffix(c3, sx, sz3);
      // chunk i + 2 has arrived, its state and what is behind it may still be on its way
      if (!state) fprt::fill_wait<COPIES>();
      else if (!halves) fprt::fill_wait<COPIES + TT::PER_WAVE>();
      else fprt::fill_wait<COPIES + 2 * TT::PER_WAVE>();
      fprt::block_sync();
      c0 = c1; c1 = c2; c2 = c3;
      c3 = walk.after(c3);
      sx = sx1;
      sz = next_z(sz);
      sp ^= 1;
    }
    fprt::fill_wait<0>();   // (nothing may arrive after the end)
    fprt::block_sync();
    return;
  }

  if (wave >= 4) {
    // ================================= score waves =================================
    const int fw = wave & 3, t = tid & 255;
    char* const Yg = reinterpret_cast<char*>(io.Y) + headB;
    // Y: rows y_row and y_row + 32, 16 bytes each, so that a store covers whole 128-byte pieces of rows
    const int y_row = t >> 3, y_piece = t & 7;
    const int q_at = Q0 + (y_piece >> 2) * FP_Q + y_row * FP_Q_LD + 16 * (y_piece & 3);
    const uint32_t y_off = (uint32_t)y_row * rowB + y_piece * 16;
    auto drain = [&](const Chunk& k, int sp) {
      const u32x4 v0 = ld128(at(q_at + sp * 4 * FP_Q)), v1 = ld128(at(q_at + sp * 4 * FP_Q + 2 * FP_Q));
      const fprt::BufView yv = fprt::make_buf(Yg + (size_t)k.row * rowB, k.L > 0 ? (uint32_t)(k.L - 1) * rowB + BV * 2 : 0u);
      // non-temporal: outputs are not read back by this launch and need not displace its inputs in the caches
      fprt::buf_store128_nt(yv, y_off, v0);
      fprt::buf_store128_nt(yv, y_off + 32 * rowB, v1);
      if (FOLD && k.sfx >= 0 && t < 8 * FP_SFX) {
        const fprt::BufView sv = fprt::make_buf(reinterpret_cast<char*>(io.Ys) + headB + (size_t)sfx_row(k) * rowB, (uint32_t)(p.Ls - 1) * rowB + BV * 2);
        fprt::buf_store128_nt(sv, y_off, ld128(at(QS0 + sp * QS_STAGE + (y_piece >> 2) * QS_HALF + y_row * FP_Q_LD + 16 * (y_piece & 3))));
      }
    };
    // The diagonal score tiles by waves 0 and 1 of the role, the other live one by wave 2, a suffix's by wave 3 (which has none otherwise)
    const bool of_suffix = FOLD && fw == 3, scores = FOLD || fw < 3, diagonal = fw < 2 || of_suffix;
    const int s_ib = fw == 0 ? 0 : fw == 1 ? 1 : REV ? 0 : 1, s_jb = diagonal ? s_ib : 1 - s_ib;   // rows of X, rows of W
    float mw[16];
    uint32_t keep[8];      // bits to keep after conversion: a masked score is cleared, so that inf or nan cannot leak through 0 * x
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
    const int x_at = of_suffix ? XS0 + TT::at(c & (FP_SFX - 1), g) : X0 + TT::at(32 * s_ib + c, g);
    const int w_at = of_suffix ? WS0 + TT::at(c & (FP_SFX - 1), g) : W0 + TT::at(32 * s_jb + c, g);
    const int p_out = (of_suffix ? PS0 : P0 + (diagonal ? s_ib : 2) * FP_P) + lane * 16, p_stage = of_suffix ? FP_P / 2 : 3 * FP_P;
    u32x4 xf[KS], wf[KS];
    // sz: FOLD, the stage in the ring of suffixes' X
    auto score_load = [&](int sx, int sz) {
      const int ow = of_suffix ? sx / (TT::BYTES / SB) : sx, ox = of_suffix ? sz / (TT::BYTES / SB) : sx;
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        wf[k] = ld128(at((w_at + ow) ^ (32 * k)));
        xf[k] = ld128(at((x_at + ox) ^ (32 * k)));
      }
    };
    auto score = [&](int sp) {
      f32x16 sc = {0};
#pragma unroll
      for (int k = 0; k < KS; ++k) sc = fprt::mfma_32x32x16_bf16(wf[k], xf[k], sc);
      // accumulator element r = 8 k + e is token 16 k + 8 (e / 4) + 4 g + e % 4 of its tile, the order the Z operands are read in
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        u32x4 d;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int r = 8 * k + 2 * e;
          d[e] = fprt::pack_bf16x2(sc[r] * mw[r], sc[r + 1] * mw[r + 1]) & keep[4 * k + e];
        }
        if (k == 0 || !of_suffix) st128(at(p_out + sp * p_stage + 1024 * k), d);
      }
    };

    Chunk c0 = walk.first(slot), cp = c0, c1 = walk.after(c0);
    cp.L = 0;
    cp.sfx = -1;
    fprt::block_sync();
    if (scores) {
      score_load(0, 0);
      score(0);
    }
    fprt::block_sync();
    int sx = 0, sz = 0, sp = 0;   // stages of chunk i
#pragma nounroll
    while (live(c1)) {
      sx = next_x(sx);
      if (FOLD) sz = next_z(sz);
      const bool now = of_suffix ? c1.sfx >= 0 : scores;
      if (now) score_load(sx, sz);
      drain(cp, sp ^ 1);
      if (now) score(sp ^ 1);
      fprt::block_sync();
      cp = c0; c0 = c1;
      c1 = walk.after(c1);
      sp ^= 1;
    }
    drain(cp, sp ^ 1);
    fprt::block_sync();
    drain(c0, sp);
    return;
  }

  // ================================= carry waves =================================
  const int ns = wave & 1, ih = wave >> 1;      // this wave: columns 32 ns .., chunk rows 32 ih ..
  // racc[a] element r is R[32 a + 16 (r / 8) + 8 g + r % 8][n], n = 32 ns + swapped(c)
  f32x16 racc[NAB];
#pragma unroll
  for (int a = 0; a < NAB; ++a) racc[a] = f32x16{0};
  const int quarter = Q0 + (2 * ih + ns) * FP_Q;

  // Elements 8 (i % 2) .. + 7 of racc[i / 2] as they are in a state tile
  auto state_piece = [&](int from, int i) {
    const int l = fprt::opaque(lane);   // (what only a change of states needs is not kept in registers between two of them)
    if (tposed) return ld128(at(from + TT::at(32 * ns + swapped(l & 31), 2 * i + (l >> 5))));
    const int row = 16 * i + 8 * (l >> 5) + ((l & 15) >> 2), q = swap2(l & 3), piece = 4 * ns + 2 * ((l >> 4) & 1) + (q >> 1), in = 8 * (q & 1);
    return joined(fprt::lds_read_tr16_b64(at(from + TT::at(row, piece) + in)), fprt::lds_read_tr16_b64(at(from + TT::at(row + 4, piece) + in)));
  };
  int states = 0;   // taken so far
  auto enter = [&]() {
    const int from = state_tile(states);
    ++states;
#pragma unroll
    for (int i = 0; i < 2 * NAB; ++i) {
      const u32x4 v = state_piece(from, i);
#pragma unroll
      for (int e = 0; e < 8; ++e) racc[i >> 1][8 * (i & 1) + e] = bf16_elem(v, e);
      if (halves) {
        const u32x4 lower = state_piece(from + TT::BYTES, i);
#pragma unroll
        for (int e = 0; e < 8; ++e) racc[i >> 1][8 * (i & 1) + e] = joined_elem(v, lower, e);
      }
    }
  };
  auto join = [&]() {
    const int from = state_tile(states);
    ++states;
#pragma unroll
    for (int i = 0; i < 2 * NAB; ++i) {
      const u32x4 v = state_piece(from, i);
#pragma unroll
      for (int e = 0; e < 8; ++e) racc[i >> 1][8 * (i & 1) + e] += bf16_elem(v, e);
    }
  };
  // ---- R -> a state matrix in global memory, 16 bytes per lane along the contiguous direction of the matrix.  R = S^T: the pieces
  // are this lane's elements.  R = S: a block of 32 rows at a time, turned in this wave's quarter of output stage sp, which nobody uses.
  const uint32_t mat_bytes = (uint32_t)p.dA * (uint32_t)p.dB * 2;
  // the two waves of a strip store half of it each
  auto leave = [&](uint16_t* dst, int sp) {
    const fprt::BufView view = fprt::make_buf(dst, mat_bytes);
    const int st = quarter + sp * 4 * FP_Q, l = fprt::opaque(lane), turn_at = (l >> 2) * FP_Q_LD + 16 * (l & 3);
    const uint32_t m_step = 2u * (tposed ? 16u : 16u * (uint32_t)io.rs_a);   // from one group of 16 rows to the next
    const uint32_t m_off = 2u * (tposed ? (uint32_t)((tile * BV + 32 * ns + swapped(l & 31)) * (int)io.rs_n + 8 * (l >> 5))
                                        : (uint32_t)((l >> 2) * (int)io.rs_a + tile * BV + 32 * ns + 8 * (l & 3)));
    auto block = [&](int a, const f32x16& acc) {
      if (tposed) {
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) fprt::buf_store128(view, m_off + (2 * a + hf) * m_step, packed(acc, hf));
        return;
      }
#pragma unroll
      for (int r = 0; r < 16; ++r)
        reinterpret_cast<u16_m*>(at(st + (16 * (r >> 3) + 8 * (l >> 5) + (r & 7)) * FP_Q_LD))[swapped(l & 31)] = float_to_bf16_bits(acc[r]);
      fprt::wave_sync();
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) fprt::buf_store128(view, m_off + (2 * a + hf) * m_step, ld128(at(st + turn_at + 16 * hf * FP_Q_LD)));
      fprt::wave_sync();
    };
#pragma unroll
    for (int a = 0; a < NAB; ++a) {
      if (a / (NAB / 2) == ih) block(a, racc[a]);
    }
  };

  Chunk cur = walk.first(slot), nxt = walk.after(cur), done = cur;
  // Operands read along the tokens: tokens 16 k + 4 g + {0..3} and + 8 of k-step k, columns in `swapped` order
  const int tr_row = 4 * g + ((lane & 15) >> 2), tr_piece = 2 * ((lane >> 4) & 1) + (swap2(lane & 3) >> 1), tr_in = 8 * (swap2(lane & 3) & 1);
  const int z_lo = TT::at(tr_row, 4 * ns + tr_piece) + tr_in, z_hi = TT::at(tr_row + 8, 4 * ns + tr_piece) + tr_in;
  const int w_lo = TT::at(tr_row, tr_piece) + tr_in, w_hi = TT::at(tr_row + 8, tr_piece) + tr_in;   // ^ 64 a: columns 32 a ..
  auto z_frag = [&](int base, int k) {
    return joined(fprt::lds_read_tr16_b64(at(base + z_lo + 16 * k * TT::PITCH)), fprt::lds_read_tr16_b64(at(base + z_hi + 16 * k * TT::PITCH)));
  };
  const int i_row = 32 * ih + c;
  const int x_at = X0 + TT::at(i_row, g);
  const bool other = REV ? ih == 0 : ih == 1;     // this row block sees the other one's tokens, too
  const float wread_fwd = io.s_read * fprt::exp2_approx((float)(REV ? CH - 1 - i_row : i_row + 1) * lg);
  const float gL_full = fprt::exp2_approx((float)CH * lg);
  const int p_at = P0 + lane * 16;
  const int y_at = quarter + c * FP_Q_LD + 16 * g;
  const int xs_at = XS0 + TT::at(c & (FP_SFX - 1), g), ys_at = QS0 + ns * QS_HALF + (c & (FP_SFX - 1)) * FP_Q_LD + 16 * g;

  fprt::block_sync();
  if (io.R0) enter();
  if (!MULTI && brings_state(cur)) join();
  u32x4 xf[KS];
#pragma unroll
  for (int k = 0; k < KS; ++k) xf[k] = ld128(at(x_at ^ (32 * k)));
  fprt::block_sync();

  int sx = 0, sz = 0, sp = 0;
  bool later = false;   // not the walk's first step
#pragma nounroll
  while (true) {
    const int L = cur.L;
    // (output stage sp: drained, not yet written again)
    if (BLOCKS && later) {
      if (!REV && io.Bout && walk.at_block_end(done)) leave(block_matrix(io.Bout, done), sp);
      if (brings_state(cur)) join();
    }
    if (MULTI && cur.first && later) {
      if (io.Rout) leave(matrix(io.Rout, cur.b - p.slots), sp);
      if (io.R0) {
        enter();
      } else {
#pragma unroll
        for (int a = 0; a < NAB; ++a) racc[a] = f32x16{0};
      }
    }
    const int pb = p_at + sp * 3 * FP_P;
    u32x4 z[4], pi[2], pj[2];   // z: the whole chunk's, for the update; of its halves the other one's scores if they are live
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      pi[k] = ld128(at(pb + ih * FP_P + 1024 * k));
      if (other) pj[k] = ld128(at(pb + 2 * FP_P + 1024 * k));
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) z[k] = z_frag(Z0 + sz, k);
    // ---- read-out of the carried state, Y^T[n][i] = sum_a R[a][n] X[i][a]
    f32x16 acc = {0};
    if (FOLD && ih == 0 && cur.sfx >= 0) {   // and the suffix's, whose rows are 0 .. 15 of a block
      const int os = sz / (TT::BYTES / SB);
      f32x16 accs = {0};
      u32x4 xs[KS];
#pragma unroll
      for (int k = 0; k < KS; ++k) xs[k] = ld128(at((xs_at + os) ^ (32 * k)));
      const u32x4 zs = z_frag(ZS0 + os, 0), ps = ld128(at(PS0 + lane * 16 + sp * (FP_P / 2)));
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        const u32x4 ra = packed(racc[k >> 1], k & 1);
        acc = fprt::mfma_32x32x16_bf16(ra, xf[k], acc);
        accs = fprt::mfma_32x32x16_bf16(ra, xs[k], accs);
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) accs[r] *= wread_fwd;
      accs = fprt::mfma_32x32x16_bf16(zs, ps, accs);
      if (c < FP_SFX) {
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) st128(at(ys_at + sp * QS_STAGE + 32 * hf), packed(accs, hf));
      }
    } else {
#pragma unroll
      for (int k = 0; k < KS; ++k) acc = fprt::mfma_32x32x16_bf16(packed(racc[k >> 1], k & 1), xf[k], acc);
    }
    fprt::sched_fence();
    // ---- what the update needs is requested, R decays, the read-out is scaled
    u32x4 wa[4][NAB];
    const int wb = WW0 + sp * TT::BYTES;
    auto request_w = [&](int k) {
#pragma unroll
      for (int a = 0; a < NAB; ++a)
        wa[k][a] = joined(fprt::lds_read_tr16_b64(at(((wb + w_lo) ^ (64 * a)) + 16 * k * TT::PITCH)),
                          fprt::lds_read_tr16_b64(at(((wb + w_hi) ^ (64 * a)) + 16 * k * TT::PITCH)));
    };
    request_w(0);
    request_w(1);
    sx = next_x(sx);
#pragma unroll
    for (int k = 0; k < KS; ++k) xf[k] = ld128(at((x_at + sx) ^ (32 * k)));
    float wread = wread_fwd;
    if (REV && L != CH) wread = io.s_read * fprt::exp2_approx((float)(i_row < L ? L - 1 - i_row : 0) * lg);
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] *= wread;
    // In the order of retention_pass_ws.h, whose waves begin with the tile that they made themselves, those of the odd column blocks the other
    // one: a call's o has the same bits whichever of the two kernels takes it
    auto other_tile = [&]() {
#pragma unroll
      for (int k = 0; k < 2; ++k) acc = fprt::mfma_32x32x16_bf16(z[REV ? 2 + k : k], pj[k], acc);   // (seen by the row block that walks later)
    };
    if (other && ns == 1) other_tile();
    if (ih == 0) {
#pragma unroll
      for (int k = 0; k < 2; ++k) acc = fprt::mfma_32x32x16_bf16(z[k], pi[k], acc);
    } else {
#pragma unroll
      for (int k = 0; k < 2; ++k) acc = fprt::mfma_32x32x16_bf16(z[2 + k], pi[k], acc);
    }
    if (other && ns == 0) other_tile();
    float gL = gL_full;
    if (L != CH) gL = fprt::exp2_approx((float)L * lg);
#pragma unroll
    for (int a = 0; a < NAB; ++a) {
#pragma unroll
      for (int r = 0; r < 16; ++r) racc[a][r] *= gL;
    }
    fprt::sched_fence();
    request_w(2);
    request_w(3);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
#pragma unroll
      for (int a = 0; a < NAB; ++a) racc[a] = fprt::mfma_32x32x16_bf16(wa[k][a], z[k], racc[a]);
    }
    // accumulator element r of Y^T is column 16 (r / 8) + 8 g + r % 8 of this wave's quarter
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) st128(at(y_at + sp * 4 * FP_Q + 32 * hf), packed(acc, hf));
    fprt::block_sync();
    if (!live(nxt)) {
      if (BLOCKS && !REV && io.Bout && walk.at_block_end(cur)) leave(block_matrix(io.Bout, cur), sp ^ 1);
      if (io.Rout) leave(matrix(io.Rout, cur.b), sp ^ 1);
      return;
    }
    if (BLOCKS) done = cur;
    cur = nxt;
    nxt = walk.after(nxt);
    sz = next_z(sz);
    sp ^= 1;
    later = true;
  }
}

template <int MODE, bool ALONE>
FP_DEVICE void retention_pass_fill(const PassArgs& p, const PassTensors& io, char* lds, int wg) {
  if constexpr (MODE != FILL_FOLD) {
    if (io.reverse) return retention_pass_fill_dir<MODE, true, ALONE>(p, io, lds, wg);
  }
  retention_pass_fill_dir<MODE, false, ALONE>(p, io, lds, wg);
}

// Whether a planned pass is a walk with folded suffixes: a forward whose suffixes fit beside a chunk, whole blocks.  The suffix walk of
// retention_pass_ws.h, a suffix one more item of it, takes the others.  Speed here over that of the walk, 16-token suffixes, inputs not in
// a cache, blocks of 16 to 64 tokens:
//                workgroups    1 block         2 blocks        4 blocks        12 blocks       32 blocks
//   64 x 64      32            1.11 to 1.12    1.27            1.46 to 1.47    1.78 to 1.81    1.94 to 2.01
//                256           1.03 to 1.13    1.06 to 1.25    1.20 to 1.41    1.12 to 1.67    1.29 to 1.85
//                1024          .99 to 1.13     1.08 to 1.27    1.21 to 1.40    1.41 to 1.69    1.23 to 1.96
//   64 x 128     128           1.11 to 1.12    1.26 to 1.28    1.43 to 1.46    1.67 to 1.76    1.87 to 1.91
//                1024          1.04 to 1.13    1.16 to 1.29    1.32 to 1.44    1.54 to 1.77    1.56 to 1.95
//   64 x 256     1024          1.07 to 1.13    1.21 to 1.30    1.37 to 1.48    1.61 to 1.73    1.72 to 1.96
// blocks of 72 to 128 tokens, 128 to 512 workgroups: 2 blocks 1.10 to 1.31, 12 blocks 1.16 to 1.61.
// B8 H12 T2048 64 x 128, blocks of 64: 76.1 us in the walk, 44.4 here (61.0 in a kernel of two roles whose rows went through registers).
inline bool pop_folds(const PassArgs& a) {
  return a.Ls > 0 && a.Ls <= FP_SFX && !a.reverse && a.dA == FP_DA && a.T == a.nblk * a.block && a.rs_n == 1;
}

}  // namespace fpk
