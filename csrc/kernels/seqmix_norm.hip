// fp32 residual stream: scaled embedding + norm, embedding + learned position, sublayer sum + residual add + next norm,
// activations, partial rotary with multi-map heads + paged K / V^T write.
//
// The residual stream x is fp32 whatever the activation type T (bf16 bits or float); norms
// are x / sqrt(mean(x^2) + eps) * (w_offset + w) with fp32 weights, rounded once to T.
#include <algorithm>
#include <initializer_list>

#include "seqmix_common.h"

namespace {

constexpr int NT = 256;

__device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) red[w] = v;
  __syncthreads();
  float t = 0.f;
#pragma unroll
  for (int i = 0; i < NT / 64; ++i) t += red[i];
  return t;
}

// x = table[token] * scale (+ add, one vector for all rows), out = norm(x).
template <typename T>
__global__ __launch_bounds__(NT) void embed_scale_norm_kernel(const int* __restrict__ tokens, const T* __restrict__ table,
                                                              float scale, const float* __restrict__ add,
                                                              const float* __restrict__ w, float eps,
                                                              float w_offset, float* __restrict__ resid,
                                                              T* __restrict__ out, int W, int vocab) {
  __shared__ float red[NT / 64];
  const int t = blockIdx.x;
  int tok = tokens[t];
  tok = tok < 0 ? 0 : (tok >= vocab ? vocab - 1 : tok);
  const T* row = table + static_cast<size_t>(tok) * W;
  float* x = resid + static_cast<size_t>(t) * W;
  float ss = 0.f;
  for (int i = threadIdx.x; i < W; i += NT) {
    float v = Elem<T>::ld(row[i]) * scale;
    if (add != nullptr) v += add[i];
    x[i] = v;
    ss += v * v;
  }
  const float r = 1.0f / sqrtf(block_sum(ss, red) / W + eps);
  T* o = out + static_cast<size_t>(t) * W;
  for (int i = threadIdx.x; i < W; i += NT) o[i] = Elem<T>::st(x[i] * r * (w_offset + w[i]));
}

// 4 consecutive elements as fp32, and back
template <typename T>
__device__ __forceinline__ f32x4 widen4(const T* p) {
  const typename Elem<T>::frag f = *reinterpret_cast<const typename Elem<T>::frag*>(p);
  f32x4 r;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if constexpr (sizeof(T) == 2) r[j] = bf2f(static_cast<bf16_t>(f[j])); else r[j] = f[j];
  }
  return r;
}
template <typename T>
__device__ __forceinline__ void narrow4(T* p, f32x4 v) {
  typename Elem<T>::frag f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if constexpr (sizeof(T) == 2) f[j] = static_cast<short>(f2bf(v[j])); else f[j] = v[j];
  }
  *reinterpret_cast<typename Elem<T>::frag*>(p) = f;
}

// The two row kernels with the row in registers (W a multiple of 4, at most 1024 CH; aligned rows): one pass over
// memory, 4 columns per access, instead of scalar accesses and a second read of the stream.  Bound by memory for
// many rows, by the latency of one row for few.  Measured (8183 rows of 2048, bf16): residual + norm of two parts 80 ->
// 39 us (14 bytes per element: 6.0 TB/s), embedding 57 -> 31; 64 rows of 4096: 22 -> 5.1, 14.6 -> 6.4.  (With the loads of a group of columns behind the
// store of the one before, the residual's were 43 and 7.7.)
template <typename T, int CH>
__global__ __launch_bounds__(NT) void embed_scale_norm_row_kernel(const int* __restrict__ tokens, const T* __restrict__ table,
                                                                  float scale, const float* __restrict__ add,
                                                                  const float* __restrict__ w, float eps, float w_offset,
                                                                  float* __restrict__ resid, T* __restrict__ out, int W, int vocab) {
  __shared__ float red[NT / 64];
  const int t = blockIdx.x, tok = min(max(tokens[t], 0), vocab - 1);
  const T* row = table + static_cast<size_t>(tok) * W;
  const size_t base = static_cast<size_t>(t) * W;
  f32x4 v[CH];
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int i = 4 * (threadIdx.x + c * NT);
    if (i < W) {
      v[c] = widen4<T>(row + i) * scale;
      if (add != nullptr) v[c] += *reinterpret_cast<const f32x4*>(add + i);
      *reinterpret_cast<f32x4*>(resid + base + i) = v[c];
#pragma unroll
      for (int j = 0; j < 4; ++j) ss += v[c][j] * v[c][j];
    }
  }
  const float r = 1.0f / sqrtf(block_sum(ss, red) / W + eps);
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int i = 4 * (threadIdx.x + c * NT);
    if (i < W) narrow4<T>(out + base + i, v[c] * r * (*reinterpret_cast<const f32x4*>(w + i) + w_offset));
  }
}

template <typename T, int CH>
__global__ __launch_bounds__(NT) void residual_norm_row_kernel(float* __restrict__ resid, const T* __restrict__ p0,
                                                               const T* __restrict__ p1, const float* __restrict__ pf,
                                                               const float* __restrict__ gate, const T* __restrict__ pg,
                                                               const float* __restrict__ w, float eps, float w_offset,
                                                               T* __restrict__ out, int W) {
  __shared__ float red[NT / 64];
  const size_t base = static_cast<size_t>(blockIdx.x) * W;
  // All loads of the row are asked for before the first is used (columns past W: the row's last four again, which are not stored).
  int at[CH];
#pragma unroll
  for (int c = 0; c < CH; ++c) at[c] = min(4 * static_cast<int>(threadIdx.x + c * NT), W - 4);
  f32x4 v[CH], s[CH], wv[CH];
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    v[c] = *reinterpret_cast<const f32x4*>(resid + base + at[c]);
    s[c] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  auto add = [&](const auto* p, float f) {
    f32x4 part[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) part[c] = widen4(p + base + at[c]);
#pragma unroll
    for (int c = 0; c < CH; ++c) s[c] += part[c] * f;
  };
  if (w != nullptr) {
#pragma unroll
    for (int c = 0; c < CH; ++c) wv[c] = *reinterpret_cast<const f32x4*>(w + at[c]);
  }
  if (p0 != nullptr && p1 != nullptr) {   // (the usual pair, without a wait between its two)
    f32x4 part[2][CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) part[0][c] = widen4(p0 + base + at[c]), part[1][c] = widen4(p1 + base + at[c]);
#pragma unroll
    for (int c = 0; c < CH; ++c) s[c] = part[0][c] + part[1][c];
  } else {
    if (p0 != nullptr) add(p0, 1.f);
    if (p1 != nullptr) add(p1, 1.f);
  }
  if (pf != nullptr) add(pf, 1.f);
  if (pg != nullptr) add(pg, 1.0f / (1.0f + expf(-gate[blockIdx.x])));
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    if (4 * (threadIdx.x + c * NT) >= W) break;
    v[c] += s[c];
    *reinterpret_cast<f32x4*>(resid + base + at[c]) = v[c];
#pragma unroll
    for (int j = 0; j < 4; ++j) ss += v[c][j] * v[c][j];
  }
  if (w == nullptr) return;
  const float r = 1.0f / sqrtf(block_sum(ss, red) / W + eps);
#pragma unroll
  for (int c = 0; c < CH; ++c)
    if (4 * (threadIdx.x + c * NT) < W) narrow4<T>(out + base + at[c], v[c] * r * (wv[c] + w_offset));
}

// x = table[token] + pos_table[position] (both of type T, summed in fp32), out = x rounded to T.
// VEC: four columns per thread (W a multiple of 4, aligned tables).
template <typename T, bool VEC>
__global__ __launch_bounds__(NT) void embed_position_kernel(const int* __restrict__ tokens, const int* __restrict__ positions,
                                                            const T* __restrict__ table, const T* __restrict__ pos_table,
                                                            float* __restrict__ resid, T* __restrict__ out, int W, int vocab,
                                                            int max_pos) {
  typedef typename Elem<T>::frag F;
  const int t = blockIdx.x;
  const int tok = min(max(tokens[t], 0), vocab - 1), pos = min(max(positions[t], 0), max_pos - 1);
  const T *a = table + static_cast<size_t>(tok) * W, *b = pos_table + static_cast<size_t>(pos) * W;
  float* x = resid + static_cast<size_t>(t) * W;
  T* o = out + static_cast<size_t>(t) * W;
  if constexpr (VEC) {
    for (int i = 4 * threadIdx.x; i < W; i += 4 * NT) {
      const F fa = *reinterpret_cast<const F*>(a + i), fb = *reinterpret_cast<const F*>(b + i);
      f32x4 v;
      F r;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (sizeof(T) == 2) {
          v[j] = bf2f(static_cast<bf16_t>(fa[j])) + bf2f(static_cast<bf16_t>(fb[j]));
          r[j] = static_cast<short>(f2bf(v[j]));
        } else {
          v[j] = fa[j] + fb[j];
          r[j] = v[j];
        }
      }
      *reinterpret_cast<f32x4*>(x + i) = v;
      *reinterpret_cast<F*>(o + i) = r;
    }
  } else {
    for (int i = threadIdx.x; i < W; i += NT) {
      const float v = Elem<T>::ld(a[i]) + Elem<T>::ld(b[i]);
      x[i] = v;
      o[i] = Elem<T>::st(v);
    }
  }
}

// x += (p0 + p1 + pf + sigmoid(gate) * pg); out = norm(x) (w == nullptr: no norm).
template <typename T>
__global__ __launch_bounds__(NT) void residual_norm_kernel(float* __restrict__ resid, const T* __restrict__ p0,
                                                           const T* __restrict__ p1, const float* __restrict__ pf,
                                                           const float* __restrict__ gate, const T* __restrict__ pg,
                                                           const float* __restrict__ w, float eps, float w_offset,
                                                           T* __restrict__ out, int W) {
  __shared__ float red[NT / 64];
  const size_t base = static_cast<size_t>(blockIdx.x) * W;
  float* x = resid + base;
  float g = 0.f;
  if (pg != nullptr) g = 1.0f / (1.0f + expf(-gate[blockIdx.x]));
  float ss = 0.f;
  for (int i = threadIdx.x; i < W; i += NT) {
    float s = 0.f;
    if (p0 != nullptr) s = Elem<T>::ld(p0[base + i]);
    if (p1 != nullptr) s += Elem<T>::ld(p1[base + i]);
    if (pf != nullptr) s += pf[base + i];
    if (pg != nullptr) s += g * Elem<T>::ld(pg[base + i]);
    const float v = x[i] + s;
    x[i] = v;
    ss += v * v;
  }
  if (w == nullptr) return;
  const float r = 1.0f / sqrtf(block_sum(ss, red) / W + eps);
  T* o = out + base;
  for (int i = threadIdx.x; i < W; i += NT) o[i] = Elem<T>::st(x[i] * r * (w_offset + w[i]));
}

// kind 0: gelu (tanh form, 0.5 (1 + tanh u) = 1 / (1 + exp(-2 u))); 1: relu squared; 2: silu.
__device__ __forceinline__ float activation(float z, int kind) {
  if (kind == 0) return z / (1.0f + expf(-1.5957691216057308f * (z + 0.044715f * z * z * z)));
  if (kind == 2) return z / (1.0f + expf(-z));
  const float p = fmaxf(z, 0.f);
  return p * p;
}

// in rows have stride `in_stride`, out is dense.
template <typename T>
__global__ __launch_bounds__(NT) void act_kernel(const T* __restrict__ in, T* __restrict__ out, int64_t rows, int n,
                                                 int64_t in_stride, int kind) {
  const int64_t total = rows * n;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * NT + threadIdx.x; i < total; i += static_cast<int64_t>(gridDim.x) * NT) {
    const int64_t r = i / n;
    const int c = static_cast<int>(i - r * n);
    out[i] = Elem<T>::st(activation(Elem<T>::ld(in[r * in_stride + c]), kind));
  }
}

// 8 columns per access, a row per grid step: no division per element.  8183 x 8192 gelu, bf16: 147 -> 66 us (4.1 TB/s).
template <typename T, int KIND>
__global__ __launch_bounds__(NT) void act_vec_kernel(const T* __restrict__ in, T* __restrict__ out, int rows, int n,
                                                     int64_t in_stride) {
  const int c = 8 * (blockIdx.x * NT + threadIdx.x);
  if (c >= n) return;
  for (int r = blockIdx.y; r < rows; r += gridDim.y) {
    const T* src = in + r * in_stride + c;
    f32x4 a = widen4<T>(src), b = widen4<T>(src + 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      a[j] = activation(a[j], KIND);
      b[j] = activation(b[j], KIND);
    }
    T* dst = out + static_cast<size_t>(r) * n + c;
    narrow4<T>(dst, a);
    narrow4<T>(dst + 4, b);
  }
}

// One block per token.  Row layout [q (n_q maps dim) | k (n_kv maps dim) | v (n_kv vdim) | ...].
// Feature i < 2 half of every map pairs with i +- half; angle = position * inv_freq[i % half] (fp32).
// K -> k_cache [NB, n_kv, BS, maps dim], V -> v_cache [NB, n_kv, vdim, BS] at `slots[t]` (slabs
// stored fragment-major when maps dim is a multiple of 4: see seqmix_attention.hip).
template <typename T>
__global__ __launch_bounds__(NT) void rope_multi_kv_kernel(const T* __restrict__ qkv, int64_t row_stride,
                                                           const int* __restrict__ positions,
                                                           const int* __restrict__ slots,
                                                           const float* __restrict__ inv_freq, int half,
                                                           T* __restrict__ q_out, T* __restrict__ k_cache,
                                                           T* __restrict__ v_cache, int n_q, int n_kv, int maps,
                                                           int dim, int vdim, int BS, int num_blocks) {
  const int t = blockIdx.x;
  const T* row = qkv + static_cast<size_t>(t) * row_stride;
  const float pos = static_cast<float>(positions[t]);
  const int slot = slots[t];
  const int blk = slot / BS, off = slot - blk * BS;
  const bool kv_ok = blk >= 0 && blk < num_blocks;
  const int qw = n_q * maps * dim, kw = n_kv * maps * dim, vw = n_kv * vdim;
  for (int idx = threadIdx.x; idx < qw + kw; idx += NT) {
    const int i = idx % dim;
    const float val = Elem<T>::ld(row[idx]);
    T o = row[idx];   // (as it is where it is not turned: st would make zeros of subnormal numbers)
    if (i < 2 * half) {
      const bool lo = i < half;
      const float other = Elem<T>::ld(row[lo ? idx + half : idx - half]);
      float s, c;
      sincosf(pos * inv_freq[lo ? i : i - half], &s, &c);
      o = Elem<T>::st(lo ? val * c - other * s : val * c + other * s);
    }
    if (idx < qw) {
      q_out[static_cast<size_t>(t) * qw + idx] = o;
    } else if (kv_ok) {
      const int kk = idx - qw;
      const int KD = maps * dim;
      const int g = kk / KD, f = kk - g * KD;
      T* slab = k_cache + (static_cast<size_t>(blk) * n_kv + g) * BS * KD;
      // KD % 4 == 0: fragment-major slab [KD / 4][BS][4] (seqmix_attention.hip); else [BS][KD]
      if ((KD & 3) == 0) slab[(static_cast<size_t>(f >> 2) * BS + off) * 4 + (f & 3)] = o;
      else slab[static_cast<size_t>(off) * KD + f] = o;
    }
  }
  if (kv_ok) {
    for (int idx = threadIdx.x; idx < vw; idx += NT) {
      const int g = idx / vdim, e = idx - g * vdim;
      T* slab = v_cache + (static_cast<size_t>(blk) * n_kv + g) * vdim * BS;
      // fragment-major slab [BS / 4][vdim][4] with the K rule above; else [vdim][BS]
      if (((maps * dim) & 3) == 0) slab[(static_cast<size_t>(off >> 2) * vdim + e) * 4 + (off & 3)] = row[qw + kw + idx];
      else slab[static_cast<size_t>(e) * BS + off] = row[qw + kw + idx];
    }
  }
}

// The same, four features per access (dim, half, vdim, the row stride multiples of 4).  A token's cosines and sines are
// computed once into LDS and serve all its heads and maps (the scalar form computed them per feature); a
// thread turns a group of four features together with the group `half` further on.  TPB tokens per workgroup: 4 (a
// wave each; four tokens on consecutive slots of one 4-key group write whole V groups) for large steps, 1 for small
// ones, whose tokens are cut into slices as long as that makes no more than 512 workgroups: a slice finds the angles again, but has one
// group of features and one value per thread (64 tokens, 32 / 8 heads of two 64-wide maps, bf16: 7.8 -> 5.9 us in four slices; scalar form
// 15.9).  8183 tokens, 16 / 4 heads: 87 -> 35 us.
constexpr int ANGLES = 128;   // pairs of a map in the LDS table

template <typename T, int TPB>
__global__ __launch_bounds__(NT) void rope_multi_kv_vec_kernel(const T* __restrict__ qkv, int64_t row_stride,
                                                               const int* __restrict__ positions, const int* __restrict__ slots,
                                                               const float* __restrict__ inv_freq, int half, T* __restrict__ q_out,
                                                               T* __restrict__ k_cache, T* __restrict__ v_cache, int n_q, int n_kv,
                                                               int maps, int dim, int vdim, int BS, int num_blocks, int n_tokens) {
  typedef typename Elem<T>::frag F;
  constexpr int TPT = NT / TPB;   // threads per token
  __shared__ __attribute__((aligned(16))) float angle[TPB][2][ANGLES];
  const int sub = threadIdx.x / TPT, tid = threadIdx.x - sub * TPT;
  const int t = blockIdx.x * TPB + sub;
  const bool live = t < n_tokens;
  const int tc = live ? t : n_tokens - 1;
  const float pos = static_cast<float>(positions[tc]);
  const int step = TPB == 1 ? TPT * gridDim.y : TPT, first = tid + (TPB == 1 ? TPT * blockIdx.y : 0);   // this slice's work
  const T* row = qkv + static_cast<size_t>(tc) * row_stride;
  const int slot = live ? slots[tc] : -1;
  const int blk = slot / BS, off = slot - blk * BS;
  const bool kv_ok = slot >= 0 && blk < num_blocks;
  const int KD = maps * dim, qw = n_q * KD, kw = n_kv * KD, vw = n_kv * vdim;
  auto put_values = [&]() {
    if (!kv_ok) return;
    for (int idx = first; idx < vw; idx += step) {
      const int g = idx / vdim, e = idx - g * vdim;
      v_cache[(static_cast<size_t>(blk) * n_kv + g) * vdim * BS + (static_cast<size_t>(off >> 2) * vdim + e) * 4 + (off & 3)] = row[qw + kw + idx];
    }
  };
  if constexpr (TPB == 1) put_values();   // (nothing to wait for but the slot)
  for (int i = tid; i < half; i += TPT) {
    float s, c;
    sincosf(pos * inv_freq[i], &s, &c);
    angle[sub][0][i] = c;
    angle[sub][1][i] = s;
  }
  __syncthreads();
  if (live) {
    const int hg = half >> 2, per = (dim - half) >> 2;   // turned groups, and groups of work, of a map
    const int jobs = (n_q + n_kv) * maps * per;
    auto place = [&](int idx) -> T* {   // (null: a key that no slot takes)
      if (idx < qw) return q_out + static_cast<size_t>(t) * qw + idx;
      const int kk = idx - qw, g = kk / KD, f = kk - g * KD;
      return kv_ok ? k_cache + (static_cast<size_t>(blk) * n_kv + g) * BS * KD + (static_cast<size_t>(f >> 2) * BS + off) * 4 : nullptr;
    };
    auto put = [&](int idx, f32x4 v) {
      if (T* p = place(idx)) narrow4<T>(p, v);
    };
    for (int job = first; job < jobs; job += step) {
      const int map = job / per, u = job - map * per;
      if (u < hg) {
        const int idx = map * dim + 4 * u;
        const f32x4 a = widen4<T>(row + idx), b = widen4<T>(row + idx + half);
        const f32x4 c = *reinterpret_cast<const f32x4*>(&angle[sub][0][4 * u]), s = *reinterpret_cast<const f32x4*>(&angle[sub][1][4 * u]);
        put(idx, a * c - b * s);
        put(idx + half, b * c + a * s);
      } else {
        const int idx = map * dim + half + 4 * u;
        if (T* p = place(idx)) *reinterpret_cast<F*>(p) = *reinterpret_cast<const F*>(row + idx);   // (as they are)
      }
    }
  }
  if constexpr (TPB == 4) {
    const int t0 = blockIdx.x * 4;
    bool group = t0 + 3 < n_tokens;   // (uniform over the workgroup)
    if (group) {
      const int s0 = slots[t0];
      group = s0 >= 0 && (s0 & 3) == 0 && s0 / BS < num_blocks && slots[t0 + 1] == s0 + 1 && slots[t0 + 2] == s0 + 2 && slots[t0 + 3] == s0 + 3;
    }
    if (group) {   // one 4-key vector per value feature
      const int s0 = slots[t0], b0 = s0 / BS, o0 = s0 - b0 * BS;
      const T* v0 = qkv + static_cast<size_t>(t0) * row_stride + qw + kw;
      for (int idx = threadIdx.x; idx < vw; idx += NT) {
        const int g = idx / vdim, e = idx - g * vdim;
        F o;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const T x = v0[static_cast<size_t>(j) * row_stride + idx];
          if constexpr (sizeof(T) == 2) o[j] = static_cast<short>(x); else o[j] = x;
        }
        *reinterpret_cast<F*>(v_cache + (static_cast<size_t>(b0) * n_kv + g) * vdim * BS + (static_cast<size_t>(o0 >> 2) * vdim + e) * 4) = o;
      }
      return;
    }
    put_values();
  }
}

bool aligned(int bytes, std::initializer_list<const void*> ptrs) {
  for (const void* p : ptrs)
    if (reinterpret_cast<uintptr_t>(p) % bytes) return false;
  return true;
}

}  // namespace

BCG_API int bcg_embed_scale_rmsnorm(const void* tokens, const void* table, float scale, const void* add, const void* w, float eps,
                                    float w_offset, void* resid, void* out, int T_, int W, int vocab, int is_f32,
                                    void* stream) {
  if (T_ <= 0) return 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (W % 4 == 0 && W <= 8192 && vocab > 0 && aligned(16, {table, add, w, resid, out})) {
#define BCG_EMBED_ROW(TYPE, CH)                                                                                                \
  embed_scale_norm_row_kernel<TYPE, CH><<<T_, NT, 0, s>>>(static_cast<const int*>(tokens), static_cast<const TYPE*>(table), scale, \
                                                          static_cast<const float*>(add), static_cast<const float*>(w), eps,   \
                                                          w_offset, static_cast<float*>(resid), static_cast<TYPE*>(out), W, vocab)
    if (is_f32) {
      if (W <= 2048) BCG_EMBED_ROW(float, 2); else if (W <= 4096) BCG_EMBED_ROW(float, 4); else BCG_EMBED_ROW(float, 8);
    } else {
      if (W <= 2048) BCG_EMBED_ROW(bf16_t, 2); else if (W <= 4096) BCG_EMBED_ROW(bf16_t, 4); else BCG_EMBED_ROW(bf16_t, 8);
    }
#undef BCG_EMBED_ROW
    return BCG_CHECK_LAUNCH();
  }
  if (is_f32)
    embed_scale_norm_kernel<float><<<T_, NT, 0, s>>>(static_cast<const int*>(tokens), static_cast<const float*>(table), scale, static_cast<const float*>(add),
                                                    static_cast<const float*>(w), eps, w_offset,
                                                    static_cast<float*>(resid), static_cast<float*>(out), W, vocab);
  else
    embed_scale_norm_kernel<bf16_t><<<T_, NT, 0, s>>>(static_cast<const int*>(tokens), static_cast<const bf16_t*>(table), scale, static_cast<const float*>(add),
                                                     static_cast<const float*>(w), eps, w_offset,
                                                     static_cast<float*>(resid), static_cast<bf16_t*>(out), W, vocab);
  return BCG_CHECK_LAUNCH();
}

BCG_API int bcg_embed_position(const void* tokens, const void* positions, const void* table, const void* pos_table, void* resid,
                               void* out, int T_, int W, int vocab, int max_pos, int is_f32, void* stream) {
  if (T_ <= 0) return 0;
  if (vocab < 1 || max_pos < 1) return -2;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int *tk = static_cast<const int*>(tokens), *ps = static_cast<const int*>(positions);
  auto al16 = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  const bool vec = W % 4 == 0 && al16(table) && al16(pos_table) && al16(resid) && al16(out);
#define BCG_EMBED(TYPE, VEC)                                                                                              \
  embed_position_kernel<TYPE, VEC><<<T_, NT, 0, s>>>(tk, ps, static_cast<const TYPE*>(table), static_cast<const TYPE*>(pos_table), \
                                                     static_cast<float*>(resid), static_cast<TYPE*>(out), W, vocab, max_pos)
  if (is_f32) {
    if (vec) BCG_EMBED(float, true); else BCG_EMBED(float, false);
  } else {
    if (vec) BCG_EMBED(bf16_t, true); else BCG_EMBED(bf16_t, false);
  }
#undef BCG_EMBED
  return BCG_CHECK_LAUNCH();
}

BCG_API int bcg_residual_add_rmsnorm32(void* resid, const void* p0, const void* p1, const void* pf, const void* gate,
                                       const void* pg, const void* w, float eps, float w_offset, void* out, int T_,
                                       int W, int is_f32, void* stream) {
  if (T_ <= 0) return 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (W > 0 && W % 4 == 0 && W <= 8192 && aligned(16, {resid, p0, p1, pf, pg, w, out})) {   // (it reads a row's last four)
#define BCG_RESIDUAL_ROW(TYPE, CH)                                                                                             \
  residual_norm_row_kernel<TYPE, CH><<<T_, NT, 0, s>>>(static_cast<float*>(resid), static_cast<const TYPE*>(p0),               \
                                                       static_cast<const TYPE*>(p1), static_cast<const float*>(pf),            \
                                                       static_cast<const float*>(gate), static_cast<const TYPE*>(pg),          \
                                                       static_cast<const float*>(w), eps, w_offset, static_cast<TYPE*>(out), W)
    if (is_f32) {
      if (W <= 2048) BCG_RESIDUAL_ROW(float, 2); else if (W <= 4096) BCG_RESIDUAL_ROW(float, 4); else BCG_RESIDUAL_ROW(float, 8);
    } else {
      if (W <= 2048) BCG_RESIDUAL_ROW(bf16_t, 2); else if (W <= 4096) BCG_RESIDUAL_ROW(bf16_t, 4); else BCG_RESIDUAL_ROW(bf16_t, 8);
    }
#undef BCG_RESIDUAL_ROW
    return BCG_CHECK_LAUNCH();
  }
  if (is_f32)
    residual_norm_kernel<float><<<T_, NT, 0, s>>>(static_cast<float*>(resid), static_cast<const float*>(p0),
                                                 static_cast<const float*>(p1), static_cast<const float*>(pf),
                                                 static_cast<const float*>(gate), static_cast<const float*>(pg),
                                                 static_cast<const float*>(w), eps, w_offset, static_cast<float*>(out), W);
  else
    residual_norm_kernel<bf16_t><<<T_, NT, 0, s>>>(static_cast<float*>(resid), static_cast<const bf16_t*>(p0),
                                                  static_cast<const bf16_t*>(p1), static_cast<const float*>(pf),
                                                  static_cast<const float*>(gate), static_cast<const bf16_t*>(pg),
                                                  static_cast<const float*>(w), eps, w_offset, static_cast<bf16_t*>(out), W);
  return BCG_CHECK_LAUNCH();
}

BCG_API int bcg_act_fn(const void* in, void* out, int64_t rows, int n, int64_t in_stride, int kind, int is_f32,
                       void* stream) {
  if (rows <= 0 || n <= 0) return 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (n % 8 == 0 && in_stride % 8 == 0 && rows < (1 << 30) && aligned(16, {in, out})) {
    const int bx = (n / 8 + NT - 1) / NT;
    const dim3 vgrid(bx, static_cast<unsigned>(std::min<int64_t>(rows, std::max<int64_t>(1, std::min(65535, 16384 / bx)))));
#define BCG_ACT(TYPE, KIND) \
  act_vec_kernel<TYPE, KIND><<<vgrid, NT, 0, s>>>(static_cast<const TYPE*>(in), static_cast<TYPE*>(out), static_cast<int>(rows), n, in_stride)
    if (is_f32) {
      if (kind == 0) BCG_ACT(float, 0); else if (kind == 2) BCG_ACT(float, 2); else BCG_ACT(float, 1);
    } else {
      if (kind == 0) BCG_ACT(bf16_t, 0); else if (kind == 2) BCG_ACT(bf16_t, 2); else BCG_ACT(bf16_t, 1);
    }
#undef BCG_ACT
    return BCG_CHECK_LAUNCH();
  }
  const int64_t total = rows * n;
  const int grid = static_cast<int>(std::min<int64_t>((total + NT - 1) / NT, 65536));
  if (is_f32)
    act_kernel<float><<<grid, NT, 0, s>>>(static_cast<const float*>(in), static_cast<float*>(out), rows, n, in_stride, kind);
  else
    act_kernel<bf16_t><<<grid, NT, 0, s>>>(static_cast<const bf16_t*>(in), static_cast<bf16_t*>(out), rows, n, in_stride, kind);
  return BCG_CHECK_LAUNCH();
}

BCG_API int bcg_rope_multi_kv_write(const void* qkv, int64_t row_stride, const void* positions, const void* slots,
                                    const void* inv_freq, int half, void* q_out, void* k_cache, void* v_cache, int T_,
                                    int n_q, int n_kv, int maps, int dim, int vdim, int BS, int num_blocks, int is_f32,
                                    void* stream) {
  if (T_ <= 0) return 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (half >= 0 && half <= ANGLES && 2 * half <= dim && half % 4 == 0 && dim % 4 == 0 && vdim % 4 == 0 && row_stride % 4 == 0 &&
      BS % 4 == 0 && aligned(16, {q_out, k_cache, v_cache}) && aligned(is_f32 ? 16 : 8, {qkv})) {
    // (groups of four features turned, or the values, of a token over the workgroups that the CUs have room for; see the kernel)
    const int work = std::max((n_q + n_kv) * maps * ((dim - half) / 4), n_kv * vdim);
    const int slices = std::max(1, std::min((work + NT - 1) / NT, 512 / T_));
#define BCG_ROPE_VEC(TYPE, TPB)                                                                                               \
  rope_multi_kv_vec_kernel<TYPE, TPB><<<dim3((T_ + TPB - 1) / TPB, TPB == 1 ? slices : 1), NT, 0, s>>>(                                                    \
      static_cast<const TYPE*>(qkv), row_stride, static_cast<const int*>(positions), static_cast<const int*>(slots),          \
      static_cast<const float*>(inv_freq), half, static_cast<TYPE*>(q_out), static_cast<TYPE*>(k_cache),                      \
      static_cast<TYPE*>(v_cache), n_q, n_kv, maps, dim, vdim, BS, num_blocks, T_)
    if (T_ >= 1024) {
      if (is_f32) BCG_ROPE_VEC(float, 4); else BCG_ROPE_VEC(bf16_t, 4);
    } else {
      if (is_f32) BCG_ROPE_VEC(float, 1); else BCG_ROPE_VEC(bf16_t, 1);
    }
#undef BCG_ROPE_VEC
    return BCG_CHECK_LAUNCH();
  }
  if (is_f32)
    rope_multi_kv_kernel<float><<<T_, NT, 0, s>>>(static_cast<const float*>(qkv), row_stride, static_cast<const int*>(positions),
                                                 static_cast<const int*>(slots), static_cast<const float*>(inv_freq), half,
                                                 static_cast<float*>(q_out), static_cast<float*>(k_cache),
                                                 static_cast<float*>(v_cache), n_q, n_kv, maps, dim, vdim, BS, num_blocks);
  else
    rope_multi_kv_kernel<bf16_t><<<T_, NT, 0, s>>>(static_cast<const bf16_t*>(qkv), row_stride, static_cast<const int*>(positions),
                                                  static_cast<const int*>(slots), static_cast<const float*>(inv_freq), half,
                                                  static_cast<bf16_t*>(q_out), static_cast<bf16_t*>(k_cache),
                                                  static_cast<bf16_t*>(v_cache), n_q, n_kv, maps, dim, vdim, BS, num_blocks);
  return BCG_CHECK_LAUNCH();
}
