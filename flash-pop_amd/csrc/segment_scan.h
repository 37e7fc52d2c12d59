// Segment scan (see ScanArgs in pass_args.h): one thread carries VEC elements of one (batch, head) state matrix through the S
// segments in fp32.  The chain over the segments is one fma per element; what bounds the launch is the latency of its loads, and
// the contributions do not depend on the chain: AHEAD of them are requested together.  A state of 64 x 128 is 1024 threads of
// eight elements, so with few streams those leave most compute units idle: threads of two elements then (scan_narrow; us a
// launch, eight -> two): B1 H12 T5003 64 x 128, 20 segments 7.7 -> 5.8; B4 H4 64 x 128, 10 blocks 7.3 -> 5.9; but B3 H8
// 128 x 128, 4 segments 4.4 -> 5.1, B2 H8 128 x 256, 8 segments 4.6 -> 6.0.  What a form does not have (lower halves, block
// states) is not in its loop: as tests at run time around every load they kept the loads apart, 8.0 us a launch at
// B2 H8 T16384 128 x 256 against 6.9 us without them.
#pragma once
#include "pass_args.h"
#include "lds_access.h"

namespace fpk {

// V 16-bit elements as one access
template <int V>
struct Packed16 {
  uint32_t d[V / 2];
};
typedef uint32_t __attribute__((may_alias)) u32_m;
template <int V>
FP_DEVICE Packed16<V> ld16s(const uint16_t* p) {
  static_assert(V == 2 || V == 8, "accesses of 4 or 16 bytes");
  Packed16<V> r;
  if constexpr (V == 2) {
    r.d[0] = *reinterpret_cast<const u32_m*>(p);
  } else {
    const u32x4 v = ld128(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) r.d[i] = v[i];
  }
  return r;
}
template <int V>
FP_DEVICE void st16s(uint16_t* p, const Packed16<V>& r) {
  if constexpr (V == 2) *reinterpret_cast<u32_m*>(p) = r.d[0];
  else st128(p, u32x4{r.d[0], r.d[1], r.d[2], r.d[3]});
}
template <int V>
FP_DEVICE float elem_of(const Packed16<V>& v, int e) {
  return __builtin_bit_cast(float, (e & 1) ? v.d[e >> 1] & 0xffff0000u : v.d[e >> 1] << 16);
}
// the float whose halves are element e of `upper` and of `lower`
template <int V>
FP_DEVICE float elem_of(const Packed16<V>& upper, const Packed16<V>& lower, int e) {
  const uint32_t u = upper.d[e >> 1], l = lower.d[e >> 1];
  return __builtin_bit_cast(float, (e & 1) ? (u & 0xffff0000u) | (l >> 16) : (u << 16) | (l & 0xffffu));
}

// LO: U and init are fp32 in two planes.  BLOCKS: block states leave or join (those of calls cut at their blocks, which keep both
// halves).
template <int VEC, int AHEAD, bool LO, bool BLOCKS>
FP_DEVICE void segment_scan_form(const ScanArgs& p) {
  const int per_mat = p.M / VEC;
  const long long item = (long long)fprt::block_index() * SCAN_THREADS + fprt::thread_index();
  if (item >= (long long)p.B * p.H * per_mat) return;
  const int piece = (int)(item % per_mat);
  const int h = (int)((item / per_mat) % p.H);
  const int b = (int)(item / ((long long)per_mat * p.H));
  const float gseg = fprt::exp2_approx((float)p.Tseg * p.log2g[h]), glast = fprt::exp2_approx((float)p.Tlast * p.log2g[h]);
  const size_t in_mat = (size_t)piece * VEC;
  float r[VEC];
  if (p.R0) {
    const Packed16<VEC> v = ld16s<VEC>(p.R0 + ((size_t)b * p.H + h) * p.M + in_mat);
#pragma unroll
    for (int e = 0; e < VEC; ++e) r[e] = elem_of(v, e);
  } else {
#pragma unroll
    for (int e = 0; e < VEC; ++e) r[e] = 0.f;
  }
  auto segment = [&](int i) { return p.reverse ? p.S - 1 - i : i; };
  const size_t step = (size_t)p.H * p.M;   // elements between the matrices of two segments, or blocks, of a sequence
  const size_t block0 = (size_t)b * p.nblk * step + (size_t)h * p.M + in_mat, matrix0 = (size_t)b * p.S * step + (size_t)h * p.M + in_mat;
  auto block = [&](int m) { return block0 + (size_t)m * step; };
  auto joins = [&](int i) { return p.blocks_in && segment(i) < p.nblk; };
  auto matrix = [&](int i) { return matrix0 + (size_t)segment(i) * step; };
  for (int i0 = 0; i0 < p.S; i0 += AHEAD) {
    Packed16<VEC> u[AHEAD], ulo[LO ? AHEAD : 1], add[BLOCKS ? AHEAD : 1];
    // (init may be U: a batch is read before its first element is written.)  Every load is issued, those beyond the last segment or
    // block on what another step reads as well: behind branches the compiler waits for each before the next (B1 H12 T5003 64 x 128,
    // 20 segments: 13.2 us a launch so, 8.7 us without; B2 H8 T16384 128 x 256, 8 segments: 8.8, 7.2).
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) {
      const int i = i0 + j < p.S ? i0 + j : p.S - 1;
      u[j] = ld16s<VEC>(p.U + matrix(i));
      if (LO) ulo[LO ? j : 0] = ld16s<VEC>(p.U_lo + matrix(i));
      if (BLOCKS) add[BLOCKS ? j : 0] = ld16s<VEC>(joins(i) ? p.blocks_in + block(segment(i)) : p.U + matrix(i));
    }
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) {
      if (i0 + j >= p.S) break;
      Packed16<VEC> o;
      auto store = [&](uint16_t* dst, auto part) {
#pragma unroll
        for (int e = 0; e < VEC / 2; ++e) o.d[e] = pack16(r[2 * e], r[2 * e + 1], part);
        st16s<VEC>(dst, o);
      };
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        if (BLOCKS && joins(i0 + j)) r[e] += elem_of(add[BLOCKS ? j : 0], e);
      }
      if constexpr (LO) {
        store(p.init + matrix(i0 + j), UpperHalf{});
        store(p.init_lo + matrix(i0 + j), LowerHalf{});
      } else {
        store(p.init + matrix(i0 + j), AsBf16{});
      }
      const float g = segment(i0 + j) == p.S - 1 ? glast : gseg;
#pragma unroll
      for (int e = 0; e < VEC; ++e) r[e] = g * r[e] + (LO ? elem_of(u[j], ulo[LO ? j : 0], e) : elem_of(u[j], e));
      if (BLOCKS && p.blocks_out && segment(i0 + j) < p.nblk) store(p.blocks_out + block(segment(i0 + j)), AsBf16{});
    }
  }
  if (p.fin) {
    Packed16<VEC> o;
#pragma unroll
    for (int e = 0; e < VEC / 2; ++e) o.d[e] = fprt::pack_bf16x2(r[2 * e], r[2 * e + 1]);
    st16s<VEC>(p.fin + ((size_t)b * p.H + h) * p.M + in_mat, o);
  }
}

// workgroups of threads of `vec` elements
inline long long scan_blocks(const ScanArgs& a, int vec) {
  return ((long long)a.B * a.H * (a.M / vec) + SCAN_THREADS - 1) / SCAN_THREADS;
}

template <int VEC, int AHEAD>
FP_DEVICE void segment_scan(const ScanArgs& p) {
  if (!p.U_lo) segment_scan_form<VEC, AHEAD, false, false>(p);
  else if (!p.blocks_in && !p.blocks_out) segment_scan_form<VEC, AHEAD, true, false>(p);
  else segment_scan_form<VEC, AHEAD, true, true>(p);
}

// Host side, shared by the GPU launcher and the CPU test harness: argument check, and whether threads of eight elements would
// leave half of the compute units without a workgroup.
inline const char* check_scan(const ScanArgs& a) {
  if (a.M % SCAN_VEC != 0 || a.B < 1 || a.S < 1 || a.H < 1 || !a.U || !a.init || !a.U_lo != !a.init_lo ||
      (!a.U_lo && (a.blocks_in || a.blocks_out)))
    return "segment scan: bad arguments";
  return scan_blocks(a, SCAN_VEC) > 0x7fffffffLL ? "segment scan: too many state matrices" : nullptr;
}
inline bool scan_narrow(const ScanArgs& a, int compute_units) { return 2 * scan_blocks(a, SCAN_VEC) < compute_units; }

}  // namespace fpk
