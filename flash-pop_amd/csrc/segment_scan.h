// Segment scan (see ScanArgs in pass_args.h): one thread carries SCAN_VEC elements of one
// (batch, head) state matrix through the S segments in fp32.  The chain over the segments is one
// fma per element; what bounds the launch is the latency of its loads (a state of 64 x 128 has 1024
// threads, so a few streams are a few dozen waves), and the contributions do not depend on the chain:
// SCAN_AHEAD of them are requested together.  What a form does not have (lower halves, block states) is not in its loop: as
// tests at run time around every load they kept the loads apart, 8.0 us a launch at B2 H8 T16384 128 x 256 against
// 6.9 us without them.
#pragma once
#include "pass_args.h"
#include "lds_access.h"

namespace fpk {

// LO: U and init are fp32 in two planes.  BLOCKS: block states leave or join (those of calls cut at their blocks, which keep both
// halves).
template <bool LO, bool BLOCKS>
FP_DEVICE void segment_scan_form(const ScanArgs& p) {
  const int per_mat = p.M / SCAN_VEC;
  const long long item = (long long)fprt::block_index() * SCAN_THREADS + fprt::thread_index();
  if (item >= (long long)p.B * p.H * per_mat) return;
  const int piece = (int)(item % per_mat);
  const int h = (int)((item / per_mat) % p.H);
  const int b = (int)(item / ((long long)per_mat * p.H));
  const float gseg = fprt::exp2_approx((float)p.Tseg * p.log2g[h]), glast = fprt::exp2_approx((float)p.Tlast * p.log2g[h]);
  const size_t in_mat = (size_t)piece * SCAN_VEC;
  float r[SCAN_VEC];
  if (p.R0) {
    const u32x4 v = ld128(p.R0 + ((size_t)b * p.H + h) * p.M + in_mat);
#pragma unroll
    for (int e = 0; e < SCAN_VEC; ++e) r[e] = bf16_elem(v, e);
  } else {
#pragma unroll
    for (int e = 0; e < SCAN_VEC; ++e) r[e] = 0.f;
  }
  auto segment = [&](int i) { return p.reverse ? p.S - 1 - i : i; };
  const size_t step = (size_t)p.H * p.M;   // elements between the matrices of two segments, or blocks, of a sequence
  const size_t block0 = (size_t)b * p.nblk * step + (size_t)h * p.M + in_mat, matrix0 = (size_t)b * p.S * step + (size_t)h * p.M + in_mat;
  auto block = [&](int m) { return block0 + (size_t)m * step; };
  auto joins = [&](int i) { return p.blocks_in && segment(i) < p.nblk; };
  auto matrix = [&](int i) { return matrix0 + (size_t)segment(i) * step; };
  for (int i0 = 0; i0 < p.S; i0 += SCAN_AHEAD) {
    u32x4 u[SCAN_AHEAD], ulo[LO ? SCAN_AHEAD : 1], add[BLOCKS ? SCAN_AHEAD : 1];
    // (init may be U: a batch is read before its first element is written.)  Every load is issued, those beyond the last segment or
    // block on what another step reads as well: behind branches the compiler waits for each before the next (B1 H12 T5003 64 x 128,
    // 20 segments: 13.2 us a launch so, 8.7 us without; B2 H8 T16384 128 x 256, 8 segments: 8.8, 7.2).
#pragma unroll
    for (int j = 0; j < SCAN_AHEAD; ++j) {
      const int i = i0 + j < p.S ? i0 + j : p.S - 1;
      u[j] = ld128(p.U + matrix(i));
      if (LO) ulo[LO ? j : 0] = ld128(p.U_lo + matrix(i));
      if (BLOCKS) add[BLOCKS ? j : 0] = ld128(joins(i) ? p.blocks_in + block(segment(i)) : p.U + matrix(i));
    }
#pragma unroll
    for (int j = 0; j < SCAN_AHEAD; ++j) {
      if (i0 + j >= p.S) break;
      u32x4 o;
      auto store = [&](uint16_t* dst, auto part) {
#pragma unroll
        for (int e = 0; e < SCAN_VEC / 2; ++e) o[e] = pack16(r[2 * e], r[2 * e + 1], part);
        st128(dst, o);
      };
#pragma unroll
      for (int e = 0; e < SCAN_VEC; ++e) {
        if (BLOCKS && joins(i0 + j)) r[e] += bf16_elem(add[BLOCKS ? j : 0], e);
      }
      if constexpr (LO) {
        store(p.init + matrix(i0 + j), UpperHalf{});
        store(p.init_lo + matrix(i0 + j), LowerHalf{});
      } else {
        store(p.init + matrix(i0 + j), AsBf16{});
      }
      const float g = segment(i0 + j) == p.S - 1 ? glast : gseg;
#pragma unroll
      for (int e = 0; e < SCAN_VEC; ++e) r[e] = g * r[e] + (LO ? joined_elem(u[j], ulo[LO ? j : 0], e) : bf16_elem(u[j], e));
      if (BLOCKS && p.blocks_out && segment(i0 + j) < p.nblk) store(p.blocks_out + block(segment(i0 + j)), AsBf16{});
    }
  }
  if (p.fin) {
    u32x4 o;
#pragma unroll
    for (int e = 0; e < SCAN_VEC / 2; ++e) o[e] = fprt::pack_bf16x2(r[2 * e], r[2 * e + 1]);
    st128(p.fin + ((size_t)b * p.H + h) * p.M + in_mat, o);
  }
}

FP_DEVICE void segment_scan(const ScanArgs& p) {
  if (!p.U_lo) segment_scan_form<false, false>(p);
  else if (!p.blocks_in && !p.blocks_out) segment_scan_form<true, false>(p);
  else segment_scan_form<true, true>(p);
}

}  // namespace fpk
