// CPU stand-in for the device primitives: one OS thread per GPU lane, pthread barriers for
// workgroup and wave synchronisation, MFMA evaluated from the documented lane layout.
// Test infrastructure only: lets the kernel body run under ASan / gdb and be compared with
// the oracle without a GPU.  Never part of the shipped library.
#pragma once
#include <pthread.h>
#include <stdint.h>
#include <unistd.h>

#include <atomic>
#include <cmath>
#include <cstring>
#include <deque>

#define FP_DEVICE inline __attribute__((always_inline))

namespace fprt {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

struct WaveShared {
  uint16_t A[64][8];
  uint16_t Bm[64][8];
  float xchg[64];
  uint16_t tr[64][4];
  pthread_barrier_t bar;
};

struct LaneCtx {
  int tid, block, grid;
  WaveShared* wave;
  pthread_barrier_t* wg_bar;
};

extern thread_local LaneCtx g_lane;

FP_DEVICE int thread_index() { return g_lane.tid; }
FP_DEVICE int block_index() { return g_lane.block; }
FP_DEVICE int grid_size() { return g_lane.grid; }
// A test can have the lanes below `threads` (above, if negative) come late out of every workgroup barrier: what the others do at once then
// comes before everything that these do.
struct Lag {
  int threads, microseconds;
};
inline Lag g_lag{0, 0};
FP_DEVICE void block_sync() {
  pthread_barrier_wait(g_lane.wg_bar);
  if (g_lag.threads != 0 && (g_lag.threads > 0 ? g_lane.tid < g_lag.threads : g_lane.tid >= -g_lag.threads)) usleep(g_lag.microseconds);
}

FP_DEVICE float bf16_to_f32(uint16_t b) {
  uint32_t u = (uint32_t)b << 16;
  float f;
  std::memcpy(&f, &u, 4);
  return f;
}

FP_DEVICE uint16_t f32_to_bf16_rne(float f) {
  uint32_t u;
  std::memcpy(&u, &f, 4);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);   // NaN stays NaN
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

FP_DEVICE f32x16 mfma_32x32x16_bf16(u32x4 a, u32x4 b, f32x16 c) {
  WaveShared* w = g_lane.wave;
  const int lane = g_lane.tid & 63;
  std::memcpy(w->A[lane], &a, 16);
  std::memcpy(w->Bm[lane], &b, 16);
  pthread_barrier_wait(&w->bar);
  const int g = lane >> 5, n = lane & 31;
  for (int r = 0; r < 16; ++r) {
    const int m = 8 * (r >> 2) + 4 * g + (r & 3);
    float acc = c[r];
    for (int k = 0; k < 16; ++k) {
      acc += bf16_to_f32(w->A[m + 32 * (k >> 3)][k & 7]) * bf16_to_f32(w->Bm[n + 32 * (k >> 3)][k & 7]);
    }
    c[r] = acc;
  }
  pthread_barrier_wait(&w->bar);
  return c;
}

FP_DEVICE uint32_t pack_bf16x2(float lo, float hi) {
  return (uint32_t)f32_to_bf16_rne(lo) | ((uint32_t)f32_to_bf16_rne(hi) << 16);
}

FP_DEVICE uint32_t lower_halves(uint32_t a, uint32_t b) { return (a & 0xffffu) | (b << 16); }
FP_DEVICE uint32_t upper_halves(uint32_t a, uint32_t b) { return (a >> 16) | (b & 0xffff0000u); }
FP_DEVICE float exp2_approx(float x) { return std::exp2(x); }
FP_DEVICE void sincos_f32(float x, float& s, float& c) { s = std::sin(x); c = std::cos(x); }
FP_DEVICE float sigmoid_f32(float x) { return 1.0f / (1.0f + std::exp(-x)); }
FP_DEVICE float rsqrt_f32(float x) { return 1.0f / std::sqrt(x); }

FP_DEVICE void sched_fence() {}
FP_DEVICE void keep(u32x4) {}
FP_DEVICE int opaque(int x) { return x; }
FP_DEVICE void pace_store(uint32_t* p, uint32_t v) { __atomic_store_n(p, v, __ATOMIC_RELAXED); }
FP_DEVICE uint32_t pace_load(const uint32_t* p) { return __atomic_load_n(p, __ATOMIC_RELAXED); }
FP_DEVICE void nap() {}
// lanes are independent OS threads here, so lane-to-lane exchange through LDS needs a real barrier
FP_DEVICE void wave_sync() { pthread_barrier_wait(&g_lane.wave->bar); }
FP_DEVICE float lane_xor(float v, int mask) {
  const int lane = g_lane.tid & 63;
  g_lane.wave->xchg[lane] = v;
  wave_sync();
  const float r = g_lane.wave->xchg[lane ^ mask];
  wave_sync();
  return r;
}

// ds_read_b64_tr_b16: within each group of 16 lanes, lane i receives element i % 4 of the four
// values read by lanes 4 e + i / 4, e = 0..3
FP_DEVICE u32x2 lds_read_tr16_b64(const uint16_t* p) {
  WaveShared* w = g_lane.wave;
  const int lane = g_lane.tid & 63;
  std::memcpy(w->tr[lane], p, 8);
  wave_sync();
  const int grp = lane & ~15, i = lane & 15;
  uint16_t out[4];
  for (int e = 0; e < 4; ++e) out[e] = w->tr[grp + 4 * e + i / 4][i % 4];
  wave_sync();
  u32x2 v;
  std::memcpy(&v, out, 8);
  return v;
}


struct BufView {
  const char* base;
  uint32_t nbytes;
};
FP_DEVICE BufView make_buf(const void* base, uint32_t nbytes) { return BufView{static_cast<const char*>(base), nbytes}; }
// What a lane has under way: copies into LDS and, counted with them, its other loads and stores.  They end in order.  A copy lands as late
// as it may, when a wait (fill_wait) is for it, and until then its place in LDS holds a pattern (nan): what reads it too early, or
// what it overwrites too early, shows.
struct UnderWay {
  char* to;   // nullptr: no copy
  u32x4 data;
};
inline thread_local std::deque<UnderWay> g_under_way;
FP_DEVICE void counted() {
  if (!g_under_way.empty()) g_under_way.push_back(UnderWay{nullptr, u32x4{0u, 0u, 0u, 0u}});   // (ahead of the first copy it makes no difference)
}
inline void land(size_t left) {
  for (; g_under_way.size() > left; g_under_way.pop_front()) {
    if (g_under_way.front().to) std::memcpy(g_under_way.front().to, &g_under_way.front().data, 16);
  }
}
FP_DEVICE u32x4 bytes_at(BufView b, uint32_t off) {
  u32x4 v = {0u, 0u, 0u, 0u};
  if ((uint64_t)off + 16 <= b.nbytes) std::memcpy(&v, b.base + off, 16);
  return v;
}
FP_DEVICE u32x4 buf_load128(BufView b, uint32_t off) {
  counted();
  return bytes_at(b, off);
}
FP_DEVICE u32x2 buf_load64(BufView b, uint32_t off) {
  counted();
  u32x2 v = {0u, 0u};
  if ((uint64_t)off + 8 <= b.nbytes) std::memcpy(&v, b.base + off, 8);
  return v;
}
FP_DEVICE void buf_store128(BufView b, uint32_t off, u32x4 v) {
  counted();
  if ((uint64_t)off + 16 <= b.nbytes) std::memcpy(const_cast<char*>(b.base) + off, &v, 16);
}
FP_DEVICE void buf_store64(BufView b, uint32_t off, u32x2 v) {
  counted();
  if ((uint64_t)off + 8 <= b.nbytes) std::memcpy(const_cast<char*>(b.base) + off, &v, 8);
}
// the non-temporal forms differ only in how the device's caches treat the data
FP_DEVICE u32x4 buf_load128_nt(BufView b, uint32_t off) { return buf_load128(b, off); }
FP_DEVICE void buf_store128_nt(BufView b, uint32_t off, u32x4 v) { buf_store128(b, off, v); }
FP_DEVICE void buf_store128_through(BufView b, uint32_t off, u32x4 v) { buf_store128(b, off, v); }

typedef BufView FillView;
FP_DEVICE FillView make_fill(const void* base, uint32_t nbytes) { return make_buf(base, nbytes); }
FP_DEVICE uint32_t uniform(uint32_t x) { return x; }
typedef char* LdsAddress;
FP_DEVICE LdsAddress lds_address(char* p) { return p; }
inline std::atomic<int> g_misaligned_fills{0};   // copies from addresses that are not multiples of their 16 bytes
template <bool ONCE, int STEP, int N>
FP_DEVICE void fill_lds(const FillView& v, const uint32_t (&off)[N], LdsAddress lds) {
  for (int u = 0; u < N; ++u) {
    if ((uint64_t)off[u] + 16 <= v.nbytes && (reinterpret_cast<uintptr_t>(v.base) + off[u]) % 16 != 0) ++g_misaligned_fills;
    char* const to = lds + STEP * u + 16 * (g_lane.tid & 63);
    std::memset(to, 0xff, 16);
    g_under_way.push_back(UnderWay{to, bytes_at(v, off[u])});
  }
}
template <int N>
FP_DEVICE void fill_wait() { land(N); }

}  // namespace fprt
