// Helpers of the fp32-stream mixer kernels (seqmix_*.hip): element traits for the two activation
// types (bf16 bits / float) and a 16 x 16 MFMA step that is the same code for both.
#pragma once

#include "common.h"

typedef short s16x4 __attribute__((ext_vector_type(4)));

template <typename T> struct Elem;
template <> struct Elem<bf16_t> {
  typedef s16x4 frag;  // 4 consecutive elements: one lane's share of a 16-deep MFMA operand
  static __device__ __forceinline__ float ld(bf16_t v) { return bf2f(v); }
  static __device__ __forceinline__ bf16_t st(float f) { return f2bf(f); }
  // finite inputs (softmax weights): the hardware's round-to-nearest-even conversion
  static __device__ __forceinline__ frag pack(float a, float b, float c, float d) {
    typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
    bf16x4 r;
    r[0] = static_cast<__bf16>(a); r[1] = static_cast<__bf16>(b);
    r[2] = static_cast<__bf16>(c); r[3] = static_cast<__bf16>(d);
    return __builtin_bit_cast(frag, r);
  }
};
template <> struct Elem<float> {
  typedef f32x4 frag;
  static __device__ __forceinline__ float ld(float v) { return v; }
  static __device__ __forceinline__ float st(float f) { return f; }
  static __device__ __forceinline__ frag pack(float a, float b, float c, float d) {
    frag r;
    r[0] = a; r[1] = b; r[2] = c; r[3] = d;
    return r;
  }
};

// Grids of the recurrences over segments: heads, segments, column blocks.  A workgroup's XCD is its index modulo 8: with the segments first, 8 of them
// put all heads of one on one XCD, and the launch ends with the longest (8 segments of 700 to 1300 tokens took as long as 8 of 1300).  The
// segments come longest first where workgroups wait for a place; where all of them run at once (`at_once`) every CU gets long and short ones instead: the heads of an
// XCD begin at different segments, every other column block walks them backwards.  (Past 64 segments in the order of the batch.)
// us, segments first and this: decays in chunks, 64 heads of 128 x 128, 8 segments of 700 to 1300 tokens 657, 560 (8 of 1000: 500), 24 of 210 to 390
// 580, 470; delta rule, 32 heads, the same 828, 760 (8 of 1000: 685) and 668, 612.
inline dim3 segment_grid(int H, int B, int Z) { return B <= 65535 ? dim3(H, B, Z) : dim3(B, H, Z); }   // (the second dimension's limit)
__device__ __forceinline__ int segment_by_length(const int* q_start, int B, int at, bool back) {
  if (back) at = B - 1 - at;
  if (B > 64) return at;
  const int lane = threadIdx.x & 63, len = lane < B ? q_start[lane + 1] - q_start[lane] : -1;
  int rank = 0;
  for (int i = 0; i < B; ++i) {
    const int other = __builtin_amdgcn_readlane(len, i);
    rank += other > len || (other == len && i < lane);
  }
  return __builtin_amdgcn_readfirstlane(__ffsll(__ballot(lane < B && rank == at)) - 1);
}
__device__ __forceinline__ void segment_of(const int* q_start, int B, bool at_once, int& b, int& h) {
  if (B <= 65535) {
    b = segment_by_length(q_start, B, at_once ? (blockIdx.y + (blockIdx.x >> 3)) % B : blockIdx.y, at_once && (blockIdx.z & 1));
    h = blockIdx.x;
  } else {
    b = blockIdx.x;
    h = blockIdx.y;
  }
}

// C[16 x 16] += A[16 x 16] B[16 x 16].  Lane l holds A[m = l % 16][k = 4 (l / 16) + j],
// B[k = 4 (l / 16) + j][n = l % 16] (j = 0..3) and C[m = 4 (l / 16) + i][n = l % 16].
// bf16: one v_mfma_f32_16x16x16_bf16.  fp32: four v_mfma_f32_16x16x4_f32 (true fp32), step j
// taking element j of every lane -- both operands use the same k order, so the sum is the same.
__device__ __forceinline__ f32x4 mma16(s16x4 a, s16x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mma16(f32x4 a, f32x4 b, f32x4 c) {
#pragma unroll
  for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], c, 0, 0, 0);
  return c;
}

// 4 consecutive elements at p[0..3]; elements at index >= n_valid read as zero.  `vec`: p is
// aligned for a vector load (the caller checked the strides); otherwise element loads.
template <typename T>
__device__ __forceinline__ typename Elem<T>::frag load_frag(const T* p, int n_valid, bool vec) {
  typedef typename Elem<T>::frag F;
  if (n_valid >= 4 && vec) return *reinterpret_cast<const F*>(p);
  F r;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    T v = j < n_valid ? p[j] : T(0);
    if constexpr (sizeof(T) == 2) r[j] = static_cast<short>(v); else r[j] = v;
  }
  return r;
}

// FULL: the caller guarantees four valid, vector-aligned elements (no branch around the load,
// so a run of fragment loads is issued back to back).
template <typename T, bool FULL>
__device__ __forceinline__ typename Elem<T>::frag load_frag_t(const T* p, int n_valid, bool vec) {
  if constexpr (FULL) return *reinterpret_cast<const typename Elem<T>::frag*>(p);
  else return load_frag<T>(p, n_valid, vec);
}

// Clamped gated unit: g = min(gate, limit), u = up clamped to +-limit, g sigmoid(1.702 g) (u + 1).
__device__ __forceinline__ float clamped_glu(float gate, float up, float limit) {
  const float g = fminf(gate, limit), u = fminf(fmaxf(up, -limit), limit);
  return g / (1.0f + expf(-1.702f * g)) * (u + 1.0f);
}

// Hidden value of a gated expert from its two products (rounded to T like a projection's output):
// act 2 silu(gate) * up, the activation rounded too; act 3 `clamped_glu`, rounded once.
template <typename T>
__device__ __forceinline__ T gated_hidden(float gate, float up, int act, float limit) {
  const float g = Elem<T>::ld(Elem<T>::st(gate)), u = Elem<T>::ld(Elem<T>::st(up));
  if (act == 3) return Elem<T>::st(clamped_glu(g, u, limit));
  return Elem<T>::st(Elem<T>::ld(Elem<T>::st(g / (1.0f + expf(-g)))) * u);
}

template <typename T>
__device__ __forceinline__ typename Elem<T>::frag zero_frag() {
  typename Elem<T>::frag r;
#pragma unroll
  for (int j = 0; j < 4; ++j) r[j] = 0;
  return r;
}
