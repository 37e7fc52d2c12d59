// Device primitives the pass kernel is written against (gfx950 / CDNA4).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define FP_DEVICE __device__ __forceinline__

namespace fprt {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

FP_DEVICE int thread_index() { return threadIdx.x; }
FP_DEVICE int block_index() { return blockIdx.x; }
FP_DEVICE int grid_size() { return gridDim.x; }
FP_DEVICE void block_sync() { __syncthreads(); }

// D = A(32x16) * B(16x32) + C, bf16 inputs, fp32 accumulate (v_mfma_f32_32x32x16_bf16).
// Lane l supplies A[l%32][8*(l/32) + e] and B[8*(l/32) + e][l%32], e = 0..7, and holds
// D[8*(r/4) + 4*(l/32) + r%4][l%32] in element r.
FP_DEVICE f32x16 mfma_32x32x16_bf16(u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0,
                                                 0, 0);
}

// Two floats -> two bf16 (round to nearest even), `lo` in bits 0..15 (v_cvt_pk_bf16_f32).
FP_DEVICE uint32_t pack_bf16x2(float lo, float hi) {
  f32x2_t f = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2_t));
}

// The lower (upper) halves of two words as one, that of `a` in bits 0..15 (v_perm_b32).
FP_DEVICE uint32_t lower_halves(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x05040100u); }
FP_DEVICE uint32_t upper_halves(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }

// 2^x for x <= 0 (v_exp_f32, ~1 ulp; results below the normal range flush to zero).
FP_DEVICE float exp2_approx(float x) { return __builtin_amdgcn_exp2f(x); }
// full-precision elementary functions for the elementwise kernels
FP_DEVICE void sincos_f32(float x, float& s, float& c) { sincosf(x, &s, &c); }
// 1 / (1 + e^-x) from the hardware's 2^x and reciprocal (v_exp_f32, v_rcp_f32: ~1 ulp each; 0 and 1
// at the far ends, where e^-x overflows or vanishes)
FP_DEVICE float sigmoid_f32(float x) { return __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-1.44269504f * x)); }
FP_DEVICE float rsqrt_f32(float x) { return 1.0f / sqrtf(x); }
// value held by lane (this lane ^ mask) of the wave; every lane of the wave has to call it
FP_DEVICE float lane_xor(float v, int mask) { return __shfl_xor(v, mask, 64); }

// Transposing LDS read (ds_read_b64_tr_b16).  Every lane passes the address of four consecutive
// 16-bit values; within each group of 16 lanes, lane i receives element i % 4 of the values read
// by lanes 4 e + i / 4, e = 0..3.  With lane 4 r + q of a group pointing at columns 4 q .. 4 q + 3 of
// row r of a row-major block of 4 rows x 16 columns, lane i gets column i of the four rows: an
// MFMA operand that runs along the rows of a row-major tile.
typedef short s16x4_t __attribute__((ext_vector_type(4)));
FP_DEVICE u32x2 lds_read_tr16_b64(const uint16_t* p) {
  return __builtin_bit_cast(
      u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)(p)));
}

// Orders LDS traffic between the lanes of one wave.  The hardware executes a wave's LDS
// instructions in order, so this only has to stop the compiler from reordering them.
FP_DEVICE void wave_sync() { __builtin_amdgcn_wave_barrier(); }

// Nothing may be moved across this point by the instruction scheduler.
FP_DEVICE void sched_fence() { __builtin_amdgcn_sched_barrier(0); }
// A value that has to be there (a load: has to have arrived) at this point.
FP_DEVICE void keep(u32x4 v) { asm volatile("" ::"v"(v)); }

// The same value, of which the compiler knows nothing: what follows from it is computed where it is used, not kept in registers
FP_DEVICE int opaque(int x) {
  asm volatile("" : "+v"(x));
  return x;
}

// Bounds-checked view of global memory (raw buffer resource): loads beyond `nbytes` return
// zero and stores beyond it are dropped by the hardware, which is how ragged chunk tails
// are handled without branches.  Offsets are bytes from `base`, below 4 GiB.
struct BufView {
  __amdgpu_buffer_rsrc_t rsrc;
};
FP_DEVICE BufView make_buf(const void* base, uint32_t nbytes) {
  return BufView{__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)nbytes, 0x00020000)};
}
FP_DEVICE u32x4 buf_load128(BufView b, uint32_t off) { return __builtin_amdgcn_raw_buffer_load_b128(b.rsrc, off, 0, 0); }
FP_DEVICE u32x2 buf_load64(BufView b, uint32_t off) { return __builtin_amdgcn_raw_buffer_load_b64(b.rsrc, off, 0, 0); }
FP_DEVICE void buf_store128(BufView b, uint32_t off, u32x4 v) { __builtin_amdgcn_raw_buffer_store_b128(v, b.rsrc, off, 0, 0); }
// the same with the non-temporal hint: data that nobody reads again soon need not stay in the caches
FP_DEVICE u32x4 buf_load128_nt(BufView b, uint32_t off) { return __builtin_amdgcn_raw_buffer_load_b128(b.rsrc, off, 0, 2); }
FP_DEVICE void buf_store128_nt(BufView b, uint32_t off, u32x4 v) { __builtin_amdgcn_raw_buffer_store_b128(v, b.rsrc, off, 0, 2); }
// ... and written through (sc1): what the L2s still hold at a kernel's end has to go out before the next launch starts (fused
// backward, B32 H4 T2048 64 x 64: 64 -> 60.5 us; no difference in launches that write little).  For stores that cover whole lines
// only: a line that leaves in parts costs far more than this saves (the forward of B8 H16 T4096 128 x 128 storing half lines at
// a time: 123 -> 185 us).
FP_DEVICE void buf_store128_through(BufView b, uint32_t off, u32x4 v) { __builtin_amdgcn_raw_buffer_store_b128(v, b.rsrc, off, 0, 2 | 16); }
FP_DEVICE void buf_store64(BufView b, uint32_t off, u32x2 v) { __builtin_amdgcn_raw_buffer_store_b64(v, b.rsrc, off, 0, 0); }

// Global memory -> LDS without a way through registers: lane l's 16 bytes at byte `off[u]` of the view land at byte 16 l from
// `lds` + STEP u, which is the same in every lane (zeros, where they are beyond the view).  Asynchronous: what it wrote may be read after
// fill_wait and a barrier.  Inline assembly, because the compiler would put a wait for every copy in flight before every LDS read
// that follows; nothing but LDS is written, so there is no register for it to lose track of.  The compiler does not see the buffer
// instructions either, so the wait states that these need are here: five behind a vector instruction (v_readfirstlane) that wrote a
// word of the view, which may be the one right before this, and one behind m0.  All copies of a view at once, so that the five are
// paid once.
struct FillView {
  u32x4 words;   // the buffer resource, uniform
};
FP_DEVICE uint32_t uniform(uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); }
FP_DEVICE FillView make_fill(const void* base, uint32_t nbytes) {
  const uint64_t p = reinterpret_cast<uint64_t>(base);
  return FillView{u32x4{uniform((uint32_t)p), uniform((uint32_t)(p >> 32) & 0xffffu), uniform(nbytes), 0x00020000u}};
}
typedef uint32_t LdsAddress;
FP_DEVICE LdsAddress lds_address(const char* p) { return uniform((uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const void*)p)); }
// ONCE: with the non-temporal hint
#define FP_COPY_FIRST(HINT) "s_mov_b32 m0, %0\n\ts_nop 3\n\tbuffer_load_dwordx4 %3, %1, 0 offen" HINT " lds"
#define FP_COPY_NEXT(OFF, HINT) "\n\ts_add_u32 m0, m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %" #OFF ", %1, 0 offen" HINT " lds"
template <bool ONCE, int STEP>
FP_DEVICE void fill_lds(const FillView& v, const uint32_t (&off)[2], LdsAddress lds) {
  if (ONCE)
    asm volatile(FP_COPY_FIRST(" nt") FP_COPY_NEXT(4, " nt")
                 ::"s"(lds), "s"(v.words), "n"(STEP), "v"(off[0]), "v"(off[1]) : "memory", "m0", "scc");
  else
    asm volatile(FP_COPY_FIRST("") FP_COPY_NEXT(4, "")
                 ::"s"(lds), "s"(v.words), "n"(STEP), "v"(off[0]), "v"(off[1]) : "memory", "m0", "scc");
}
template <bool ONCE, int STEP>
FP_DEVICE void fill_lds(const FillView& v, const uint32_t (&off)[8], LdsAddress lds) {
  static_assert(!ONCE, "not with the hint");
  asm volatile(FP_COPY_FIRST("") FP_COPY_NEXT(4, "") FP_COPY_NEXT(5, "") FP_COPY_NEXT(6, "") FP_COPY_NEXT(7, "") FP_COPY_NEXT(8, "")
               FP_COPY_NEXT(9, "") FP_COPY_NEXT(10, "")
               ::"s"(lds), "s"(v.words), "n"(STEP), "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "v"(off[4]), "v"(off[5]),
               "v"(off[6]), "v"(off[7]) : "memory", "m0", "scc");
}
#undef FP_COPY_FIRST
#undef FP_COPY_NEXT
// Until at most N of this wave's loads, copies and stores are still under way (they end in order).
template <int N>
FP_DEVICE void fill_wait() {
  static_assert(N >= 0 && N < 64, "six bits");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// A word that another workgroup of the same launch polls (relaxed, device scope), and a short sleep between polls.
FP_DEVICE void pace_store(uint32_t* p, uint32_t v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
FP_DEVICE uint32_t pace_load(const uint32_t* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
FP_DEVICE void nap() { __builtin_amdgcn_s_sleep(8); }

}  // namespace fprt
