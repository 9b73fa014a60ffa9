// FP8 (OCP e4m3fn, gfx950) activation quantisation for the fp8 projection path.
//
// Row-wise dynamic scaling: scale[r] = max|y[r,:]| / 448, q = y / scale
// (clamped to +-448, round-to-nearest-even by v_cvt_pk_fp8_f32).  The GEMM is
// hipBLASLt's fp8 kernel through torch._scaled_mm with row-wise scales on both
// operands (weights are quantised per output channel at load time), running at
// ~2x the bf16 rate.  The quantisation is fused into the producers so the fp8
// path adds no extra pass over the activations:
//   add_rmsnorm_fp8 : residual add + RMSNorm (bf16-rounded, as the bf16 path) + quant
//                     (also: plain RMSNorm + quant after a residual GEMM epilogue, and the
//                     embedding gather + RMSNorm + quant of the first layer)
//   silu_mul_fp8    : SiLU(gate) * up (bf16-rounded) + quant
//   quant_fp8       : stand-alone (attention output before o_proj)
// One workgroup per row; the row max is a wave64 shuffle reduction plus one partial per wave in
// LDS.  Rows are held in registers between the reduction and the store (one pass over memory).  A step of
// few rows is the latency of one row: 1024 threads per row there (up to WIDE_T rows; 20 rows of 2 x 16384 silu_mul: 18.1
// -> 5.0 us (6.7 with a division per value for the quotients too), 6144-wide norm 7.6 -> 4.9), 256 beyond, where several rows share a CU.

#include "common.h"

BCG_API int bcg_quant_fp8(const void* x, void* q, float* scale, int T, int K, hipStream_t stream);

namespace {

constexpr int QT = 256;
constexpr int WIDE = 1024, WIDE_T = 256;   // threads of a row in steps of up to WIDE_T rows
constexpr float FP8_MAX = 448.f;
constexpr int NORM_MAX_CHUNK = 4;  // H <= 256 * 8 * 4

__device__ __forceinline__ uint32_t pack4_fp8(float a, float b, float c, float d) {
  const uint32_t lo = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
  return __builtin_amdgcn_cvt_pk_fp8_f32(c, d, lo, true);
}

__device__ __forceinline__ float clampq(float v) { return fminf(fmaxf(v, -FP8_MAX), FP8_MAX); }

template <int TH = QT>
__device__ __forceinline__ float block_max(float v, float* red) {
  v = wave_max(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float m = red[0];
#pragma unroll
  for (int i = 1; i < TH / WAVE; ++i) m = fmaxf(m, red[i]);
  return m;
}

__device__ __forceinline__ float row_scale(float amax) { return fmaxf(amax, 1e-12f) / FP8_MAX; }

// A row's scale and what its values are divided with: a division is ten instructions, and a step of few rows is one workgroup's arithmetic per
// row, so the row divides once and a value takes the reciprocal and one residual step, three instructions.  The quotient has the
// division's bits (for every mantissa of a bf16 maximum and value): values and maxima of 8 bits make many
// quotients exact ties between two of e4m3's values (up to 1 % of a row), which a bare reciprocal rounds either way, a whole e4m3 step apart.
struct RowScale {
  float s, inv, back;
  __device__ explicit RowScale(float amax) : s(row_scale(amax)), inv(1.f / s), back(isinf(s) ? 0.f : s) {}   // (over infinity finite values are 0)
  __device__ float over(float y) const {
    const float q = y * inv;
    return __builtin_fmaf(-__builtin_fmaf(q, back, -y), inv, q);   // (in these signs zeros keep theirs)
  }
};

// store 8 quantised values (8 bytes)
__device__ __forceinline__ void store_q8(uint8_t* dst, const float (&y)[8], const RowScale& r) {
  uint2 p;
  p.x = pack4_fp8(clampq(r.over(y[0])), clampq(r.over(y[1])), clampq(r.over(y[2])), clampq(r.over(y[3])));
  p.y = pack4_fp8(clampq(r.over(y[4])), clampq(r.over(y[5])), clampq(r.over(y[6])), clampq(r.over(y[7])));
  *reinterpret_cast<uint2*>(dst) = p;
}

__global__ __launch_bounds__(QT) void quant_fp8_kernel(const bf16_t* __restrict__ x, uint8_t* __restrict__ q,
                                                       float* __restrict__ scale, int K) {
  __shared__ float red[QT / WAVE];
  const size_t base = static_cast<size_t>(blockIdx.x) * K;
  const int nvec = K / 8;
  float amax = 0.f;
  for (int vi = threadIdx.x; vi < nvec; vi += QT) {
    const u16x8 v = *reinterpret_cast<const u16x8*>(x + base + vi * 8);
#pragma unroll
    for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(bf2f(v[j])));
  }
  const RowScale r(block_max(amax, red));
  if (threadIdx.x == 0) scale[blockIdx.x] = r.s;
  for (int vi = threadIdx.x; vi < nvec; vi += QT) {
    const u16x8 v = *reinterpret_cast<const u16x8*>(x + base + vi * 8);
    float y[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) y[j] = bf2f(v[j]);
    store_q8(q + base + vi * 8, y, r);
  }
}

// has_residual: 0 = residual <- x, 1 = residual <- residual + x, 2 = plain RMSNorm of x (the
// residual stream was updated by the GEMM epilogue that produced x: nothing written back).
// gather != nullptr: x row = table row gather[row] (the embedding lookup fused in).
template <int TH, int CHUNKS>
__global__ __launch_bounds__(TH) void add_rmsnorm_fp8_kernel(
    const bf16_t* __restrict__ x, bf16_t* __restrict__ residual, const bf16_t* __restrict__ w,
    uint8_t* __restrict__ q, float* __restrict__ scale, int H, float eps, int has_residual,
    const int* __restrict__ gather) {
  __shared__ float red[TH / WAVE];
  const int tid = threadIdx.x;
  const int nvec = H / 8;
  const size_t base = static_cast<size_t>(blockIdx.x) * H;
  // x row: the gathered table row (embedding lookup fused in) or this block's row
  const bf16_t* __restrict__ xr = gather ? x + static_cast<size_t>(gather[blockIdx.x]) * H : x + base;
  // (all loads before the first use, as the bf16 form)
  u16x8 xv[CHUNKS], rv[CHUNKS], wv[CHUNKS];
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int at = min(tid + c * TH, nvec - 1) * 8;
    xv[c] = *reinterpret_cast<const u16x8*>(xr + at);
    wv[c] = *reinterpret_cast<const u16x8*>(w + at);
  }
  if (has_residual == 1) {
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) rv[c] = *reinterpret_cast<const u16x8*>(residual + base + min(tid + c * TH, nvec - 1) * 8);
  }
  float v[CHUNKS][8];
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int vi = tid + c * TH;
    if (vi < nvec) {
      u16x8 nr;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float f = bf2f(xv[c][j]);
        if (has_residual == 1) f += bf2f(rv[c][j]);
        nr[j] = has_residual == 1 ? f2bf(f) : xv[c][j];
        f = bf2f(nr[j]);
        v[c][j] = f;
        ss += f * f;
      }
      if (has_residual != 2) *reinterpret_cast<u16x8*>(residual + base + vi * 8) = nr;
    }
  }
  ss = wave_sum(ss);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  float tot = 0.f;
#pragma unroll
  for (int i = 0; i < TH / WAVE; ++i) tot += red[i];
  const float rstd = rsqrtf(tot / H + eps);
  __syncthreads();  // red[] is reused by block_max
  float amax = 0.f;
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int vi = tid + c * TH;
    if (vi < nvec) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        v[c][j] = bf2f(f2bf(v[c][j] * rstd * bf2f(wv[c][j])));  // the bf16 path's rounding
        amax = fmaxf(amax, fabsf(v[c][j]));
      }
    }
  }
  const RowScale r(block_max<TH>(amax, red));
  if (tid == 0) scale[blockIdx.x] = r.s;
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int vi = tid + c * TH;
    if (vi < nvec) store_q8(q + base + vi * 8, v[c], r);
  }
}

__device__ __forceinline__ void silu8(const bf16_t* g, float (&y)[8], int I) {
  const u16x8 gv = *reinterpret_cast<const u16x8*>(g);
  const u16x8 uv = *reinterpret_cast<const u16x8*>(g + I);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float a = bf2f(gv[j]);
    y[j] = bf2f(f2bf(a / (1.f + __expf(-a)) * bf2f(uv[j])));
  }
}

template <int TH, int CHUNKS>
__global__ __launch_bounds__(TH) void silu_mul_fp8_kernel(const bf16_t* __restrict__ gu, uint8_t* __restrict__ q,
                                                          float* __restrict__ scale, int I) {
  __shared__ float red[TH / WAVE];
  const bf16_t* row = gu + static_cast<size_t>(blockIdx.x) * 2 * I;
  uint8_t* qrow = q + static_cast<size_t>(blockIdx.x) * I;
  const int nvec = I / 8;
  float amax = 0.f, y[CHUNKS][8];
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int vi = threadIdx.x + c * TH;
    if (vi < nvec) {
      silu8(row + vi * 8, y[c], I);
#pragma unroll
      for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(y[c][j]));
    }
  }
  const RowScale r(block_max<TH>(amax, red));
  if (threadIdx.x == 0) scale[blockIdx.x] = r.s;
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int vi = threadIdx.x + c * TH;
    if (vi < nvec) store_q8(qrow + vi * 8, y[c], r);
  }
}

// Rows too long for the registers: the row is read again (from L2) for the store.
__global__ __launch_bounds__(QT) void silu_mul_fp8_long_kernel(const bf16_t* __restrict__ gu, uint8_t* __restrict__ q,
                                                               float* __restrict__ scale, int I) {
  __shared__ float red[QT / WAVE];
  const bf16_t* row = gu + static_cast<size_t>(blockIdx.x) * 2 * I;
  uint8_t* qrow = q + static_cast<size_t>(blockIdx.x) * I;
  const int nvec = I / 8;
  float amax = 0.f;
  for (int vi = threadIdx.x; vi < nvec; vi += QT) {
    float y[8];
    silu8(row + vi * 8, y, I);
#pragma unroll
    for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(y[j]));
  }
  const RowScale r(block_max(amax, red));
  if (threadIdx.x == 0) scale[blockIdx.x] = r.s;
  for (int vi = threadIdx.x; vi < nvec; vi += QT) {
    float y[8];
    silu8(row + vi * 8, y, I);
    store_q8(qrow + vi * 8, y, r);
  }
}

int launch_norm(const void* x, void* residual, const void* w, void* q, float* scale, int T, int H, float eps, int has_residual,
                const int* gather, hipStream_t stream) {
  if (H == 0) return bcg_quant_fp8(x, q, scale, T, H, stream);   // (scales of nothing; the kernel reads a row's last vector)
#define BCG_NORM_FP8(TH, CH)                                                                                                  \
  hipLaunchKernelGGL((add_rmsnorm_fp8_kernel<TH, CH>), dim3(T), dim3(TH), 0, stream, static_cast<const bf16_t*>(x),            \
                     static_cast<bf16_t*>(residual), static_cast<const bf16_t*>(w), static_cast<uint8_t*>(q), scale, H, eps,  \
                     has_residual, gather)
  if (T <= WIDE_T) BCG_NORM_FP8(WIDE, 1);   // (H <= 8192 = 1024 * 8)
  else BCG_NORM_FP8(QT, NORM_MAX_CHUNK);
#undef BCG_NORM_FP8
  return BCG_CHECK_LAUNCH();
}

}  // namespace

BCG_API int bcg_quant_fp8(const void* x, void* q, float* scale, int T, int K, hipStream_t stream) {
  if (K % 8 || T <= 0) return -2;
  hipLaunchKernelGGL(quant_fp8_kernel, dim3(T), dim3(QT), 0, stream, static_cast<const bf16_t*>(x),
                     static_cast<uint8_t*>(q), scale, K);
  return BCG_CHECK_LAUNCH();
}

BCG_API int bcg_add_rmsnorm_fp8(const void* x, void* residual, const void* w, void* q, float* scale, int T, int H,
                                float eps, int has_residual, hipStream_t stream) {
  if (H % 8 || H > QT * 8 * NORM_MAX_CHUNK || T <= 0 || has_residual < 0 || has_residual > 2) return -2;
  return launch_norm(x, residual, w, q, scale, T, H, eps, has_residual, nullptr, stream);
}

// residual[t] <- table[tokens[t]]; (q, scale)[t] <- fp8(rmsnorm(residual[t]) * w): the fp8 path's
// first layer input in one pass.  Token ids must be < vocab (checked by their producers).
BCG_API int bcg_embed_rmsnorm_fp8(const int* tokens, const void* table, const void* w, void* residual, void* q,
                                  float* scale, int T, int H, float eps, hipStream_t stream) {
  if (H % 8 || H > QT * 8 * NORM_MAX_CHUNK || T <= 0) return -2;
  return launch_norm(table, residual, w, q, scale, T, H, eps, 0, tokens, stream);
}

BCG_API int bcg_silu_mul_fp8(const void* gu, void* q, float* scale, int T, int I, hipStream_t stream) {
  if (I % 8 || T <= 0) return -2;
#define BCG_SILU_FP8(KERNEL, TH) \
  hipLaunchKernelGGL((KERNEL), dim3(T), dim3(TH), 0, stream, static_cast<const bf16_t*>(gu), static_cast<uint8_t*>(q), scale, I)
  if (I <= 8 * WIDE * 2) {
    if (T <= WIDE_T) BCG_SILU_FP8((silu_mul_fp8_kernel<WIDE, 2>), WIDE);
    else if (I <= 8 * QT * 4) BCG_SILU_FP8((silu_mul_fp8_kernel<QT, 4>), QT);
    else BCG_SILU_FP8((silu_mul_fp8_kernel<QT, 8>), QT);
  } else {
    BCG_SILU_FP8(silu_mul_fp8_long_kernel, QT);
  }
#undef BCG_SILU_FP8
  return BCG_CHECK_LAUNCH();
}
