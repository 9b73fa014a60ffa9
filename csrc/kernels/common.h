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

// Parts that several workgroups leave in memory for the one of them that arrives last, without L2 maintenance (gemm.hip): write-through stores,
// drained by every wave, one ticket, loads that pass the L2 too.
__device__ __forceinline__ void store_through(float* p, float v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ float load_through(const float* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// Whether this workgroup is the last of n that leave parts under `counter` (zero before and after).  flag: an int in LDS; every thread calls.
__device__ __forceinline__ bool last_of(int* counter, int n, int* flag) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    const int last = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == n - 1;
    if (last) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *flag = last;
  }
  __syncthreads();
  const bool last = *flag != 0;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");   // (no instruction: keeps the loads behind it)
  return last;
}

// Parts of the rows of a decode step whose pairs (row, kv head) are a workgroup each.  A row is cut where it is long by itself and in its step: past `one`
// chunks into as many parts as its share of the step's chunks is of `ways` workgroups, `parts` and one for `each` chunks at the most.  So rows of equal
// lengths are cut as far as CUs are idle, and a long row beside short ones is not walked by one workgroup per head while the others are idle; the
// lengths decide, not the room in the block table.  Those beyond a pair's first are workgroups of their own, `ways` at most in all, which find their row by
// a scan over the rows (1 to 2 us, also where there is none for them: beside the others' work); a row of up to `one` chunks pays nothing.  The part that
// arrives last adds them up: as long as a merge launch where rows are cut (1 us longer for one row of 2000 tokens), nothing where none is.
// us, parts by the number of pairs and the table's width, merged by a launch -> this (before both: rotary launch, items or stream of 256 tokens, merge).  Heads
// of 128, 8 kv heads: a row of 16000 tokens beside 9 of 400 58 -> 25 (34), beside 32 153 -> 34 (42), beside 447 of 60 222 -> 67 (73); 10 of 400 in a table for
// 8192 11.6 -> 10.7 (16.7), 10 of 1100 16.9 -> 16.6 (22.2); heads of 64: 4 of 500 in a table for 8192 8.0 -> 6.0 (10.7).  Two 64-wide maps over 128, 8 kv heads: 16000
// beside 32 of 400 170 -> 37 (117), 1 of 40 in a table for 8192 18.8 -> 6.3 (10.5), 2 of 2000 18.1 -> 15.5 (24.1).
struct PartRule {
  int parts, one, each;   // each 0: every row in `parts`
  int ways;               // workgroups that the step's chunks are shared among
  int extra;              // workgroups beside the pairs' own
};
struct Share {
  int row, part, n;   // (row < 0: none)
  int first;          // of the extra workgroups of one of the row's pairs
};
// Where workgroup `id` of pairs + extra stands: the pairs' own first where they leave places for others (cut rows' parts then come to idle CUs before the
// extra ones without a row do: 80 pairs of 6000 tokens 55 us, 68 the other way round), else the extra ones, so that long rows do not begin last.  own: a
// pair, else an extra one, `at`-th of its kind.
struct Place { bool own; int at; };
__device__ __forceinline__ Place place_of(const PartRule& r, int id, int pairs) {
  if (pairs <= 352) return id < pairs ? Place{true, id} : Place{false, id - pairs};
  return id < r.extra ? Place{false, id} : Place{true, id - r.extra};
}
// The share of row `row`'s own workgroup (part 0), or with row < 0 of extra workgroup `extra` of a pair's column; chunks(i): of row i.  Whole waves call.
template <typename Chunks>
__device__ __forceinline__ Share find_share(const PartRule& r, int rows, int pairs_per_row, int row, int extra, Chunks chunks) {
  const int lane = threadIdx.x & 63;
  int sum = 0, longest = 0;
  if (r.each > 0) {
    for (int i = lane; i < rows; i += WAVE) {
      const int all = chunks(i);
      sum += all;
      longest = max(longest, all);
    }
    if (__ballot(longest > r.one) == 0) return Share{-1, 0, 1, 0};   // (an extra workgroup: nothing is cut)
  }
  const float per_chunk = r.ways / (static_cast<float>(wave_sum(sum)) * pairs_per_row);
  int before = 0;
  for (int i0 = 0; i0 < rows; i0 += WAVE) {
    int n = 1;
    if (i0 + lane < rows) {
      const int all = chunks(i0 + lane);
      if (r.each == 0) n = r.parts;
      else if (all > r.one) n = max(1, min(min(r.parts, (all + r.each - 1) / r.each), static_cast<int>(all * per_chunk)));
    }
    int end = n - 1;
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1) {
      const int u = __shfl_up(end, o, WAVE);
      if (lane >= o) end += u;
    }
    end += before;
    const unsigned long long here = __ballot(row >= 0 ? i0 + lane == row : end - (n - 1) <= extra && extra < end);
    if (here != 0) {
      const int at = __ffsll(here) - 1, parts = __builtin_amdgcn_readlane(n, at), first = __builtin_amdgcn_readlane(end, at) - (parts - 1);
      return Share{i0 + at, row >= 0 ? 0 : extra - first + 1, parts, first};
    }
    before = __builtin_amdgcn_readlane(end, WAVE - 1);
  }
  return Share{-1, 0, 1, 0};
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
