// Shared helpers for the BCG MI355X (gfx950 / CDNA4) kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#define BCG_API extern "C" __attribute__((visibility("default")))

typedef uint16_t bf16_t;                                       // raw bf16 bits
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));    // MFMA operand
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int WAVE = 64;

__device__ __forceinline__ float bf2f(bf16_t v) { return __uint_as_float(static_cast<uint32_t>(v) << 16); }

// round to nearest even by the hardware's conversion (one instruction; in integer arithmetic it was seven, a good part of what a
// pass over a stream computes).  Infinities and NaN stay what they are, subnormal numbers are zeros as behind every operation of this build (so a
// value that is only passed on is copied as it is, not taken through here).
__device__ __forceinline__ bf16_t f2bf(float f) { return __builtin_bit_cast(bf16_t, static_cast<__bf16>(f)); }

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, WAVE);
  return v;
}

template <typename T>
__device__ __forceinline__ T wave_max(T v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, WAVE));
  return v;
}

__device__ __forceinline__ uint32_t fmix32(uint32_t h) {
  h ^= h >> 16;
  h *= 0x85ebca6bu;
  h ^= h >> 13;
  h *= 0xc2b2ae35u;
  h ^= h >> 16;
  return h;
}

typedef uint32_t quad_u32x4 __attribute__((ext_vector_type(4)));

// out[j] of lane q of a quad = in[q] of the quad's lane j: from loads in which a quad reads 64 bytes of one row (in[i]: row i of the
// quad) to lane q holding row q.  A CU takes in 117 B/ns out of L2 where four neighbouring lanes read 64 bytes of a row, 36 where they
// read 16 bytes of four rows.  One select per dword and stage takes its other side from the neighbour (hipcc makes branches
// of it).  A VALU result is read through DPP, and by a matrix instruction, two wait states later at the earliest: hipcc
// knows that of its own instructions only, so the block keeps the distance on both sides.
__device__ __forceinline__ void quad_transpose(const quad_u32x4 (&in)[4], quad_u32x4 (&out)[4]) {
  const uint64_t odd = 0xaaaaaaaaaaaaaaaaull, even = ~odd, hi = 0xccccccccccccccccull, lo = ~hi;
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    uint32_t t0, t1, t2, t3, o0, o1, o2, o3;
    asm("s_nop 1\n\t"
        "s_mov_b64 vcc, %[odd]\n\t"
        "v_cndmask_b32_dpp %[t1], %[a], %[b], vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_cndmask_b32_dpp %[t3], %[c], %[d], vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "s_mov_b64 vcc, %[even]\n\t"
        "v_cndmask_b32_dpp %[t0], %[b], %[a], vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_cndmask_b32_dpp %[t2], %[d], %[c], vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "s_mov_b64 vcc, %[hi]\n\t"
        "s_nop 0\n\t"
        "v_cndmask_b32_dpp %[o3], %[t1], %[t3], vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_cndmask_b32_dpp %[o2], %[t0], %[t2], vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "s_mov_b64 vcc, %[lo]\n\t"
        "v_cndmask_b32_dpp %[o1], %[t3], %[t1], vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_cndmask_b32_dpp %[o0], %[t2], %[t0], vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        : [t0] "=&v"(t0), [t1] "=&v"(t1), [t2] "=&v"(t2), [t3] "=&v"(t3), [o0] "=&v"(o0), [o1] "=&v"(o1), [o2] "=&v"(o2), [o3] "=&v"(o3)
        : [a] "v"(in[0][d]), [b] "v"(in[1][d]), [c] "v"(in[2][d]), [d] "v"(in[3][d]), [odd] "s"(odd), [even] "s"(even), [hi] "s"(hi),
          [lo] "s"(lo)
        : "vcc");
    out[0][d] = o0, out[1][d] = o1, out[2][d] = o2, out[3][d] = o3;
  }
}


#define BCG_CHECK_LAUNCH() (hipGetLastError() == hipSuccess ? 0 : -1)
