// Row-wise RMSNorm with fused residual add, and SiLU-and-mul.
//
// add_rmsnorm: one workgroup per row; every thread owns up to MAX_CHUNK 16-byte chunks (8 bf16) kept in registers, so the row
// is read once and written twice (residual + normed) -- the HBM minimum for the fused op.  Sum of squares: wave
// shuffle reduce, then the waves' partials via LDS.  Up to FEW_ROWS rows a launch is the latency of one row: one chunk a thread (101 rows of
// 4096: 5.2 -> 4.9 us, 20 of 6144 6.7 -> 4.8); beyond, 256 threads a row and as many chunks as it has (4449 rows of 4096 19.4 -> 17.8, 4.1 TB/s).
//
// embed_rmsnorm (K-EMB fused with layer 0's input norm): the same row kernel
// reading row tokens[t] of the embedding table, so the embedding never makes
// a separate HBM round trip: residual <- E[tok], out <- rmsnorm(E[tok]) * w.
//
// silu_mul: grid-stride over 8-element vectors of [T, 2I] -> [T, I].

#include "common.h"

namespace {

constexpr int NORM_THREADS = 256;
constexpr int MAX_CHUNK = 4;  // H <= 256 * 8 * 4 = 8192
constexpr int FEW_ROWS = 256;

// All loads of a row are asked for before the first is used, the weights' too (vectors past H: the last one again, which counts for nothing and is
// not stored).
template <int TH, int CHUNKS>
__global__ __launch_bounds__(TH) void add_rmsnorm_kernel(
    const bf16_t* __restrict__ x, bf16_t* __restrict__ residual, const bf16_t* __restrict__ w,
    bf16_t* __restrict__ out, int H, float eps, int has_residual, const int* __restrict__ gather) {
  const int row = blockIdx.x;
  const int tid = threadIdx.x;
  const int nvec = H / 8;
  const size_t base = static_cast<size_t>(row) * H;
  // x row: table row gather[row] (embedding) or row `row` -- its own pointer, indexed from 0
  const bf16_t* __restrict__ xr = gather ? x + static_cast<size_t>(gather[row]) * H : x + base;
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
        f = bf2f(nr[j]);  // normalise the value actually stored (matches the reference)
        v[c][j] = f;
        ss += f * f;
      }
      // mode 2 = plain RMSNorm of x (the residual stream was already updated by the
      // GEMM epilogue that produced x): nothing to write back
      if (has_residual != 2) *reinterpret_cast<u16x8*>(residual + base + vi * 8) = nr;
    }
  }
  __shared__ float partial[TH / WAVE];
  ss = wave_sum(ss);
  if ((tid & 63) == 0) partial[tid >> 6] = ss;
  __syncthreads();
  float tot = 0.f;
#pragma unroll
  for (int i = 0; i < TH / WAVE; ++i) tot += partial[i];
  const float inv = rsqrtf(tot / H + eps);
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int vi = tid + c * TH;
    if (vi < nvec) {
      u16x8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = f2bf(v[c][j] * inv * bf2f(wv[c][j]));
      *reinterpret_cast<u16x8*>(out + base + vi * 8) = o;
    }
  }
}

// A step of few rows is the latency of one row: a vector per thread there; several rows share a CU beyond.
int launch_norm(const void* x, void* residual, const void* w, void* out, int T, int H, float eps, int has_residual, const int* gather,
                hipStream_t stream) {
  if (H == 0) return 0;   // (the kernel reads a row's last vector)
#define BCG_NORM(TH, CH)                                                                                                    \
  hipLaunchKernelGGL((add_rmsnorm_kernel<TH, CH>), dim3(T), dim3(TH), 0, stream, static_cast<const bf16_t*>(x),              \
                     static_cast<bf16_t*>(residual), static_cast<const bf16_t*>(w), static_cast<bf16_t*>(out), H, eps, has_residual, gather)
  if (T <= FEW_ROWS && H > 4096) BCG_NORM(1024, 1);
  else if (T <= FEW_ROWS && H > 2048) BCG_NORM(512, 1);
  else if (H <= 2048) BCG_NORM(NORM_THREADS, 1);
  else if (H <= 4096) BCG_NORM(NORM_THREADS, 2);
  else if (H <= 6144) BCG_NORM(NORM_THREADS, 3);
  else BCG_NORM(NORM_THREADS, MAX_CHUNK);
#undef BCG_NORM
  return BCG_CHECK_LAUNCH();
}

// One 16-B vector of gate + up per thread and grid row-major over [T, I/8]: 32-bit
// index math (a 64-bit div/mod per element was the kernel's main cost), fast exp.
__global__ __launch_bounds__(256) void silu_mul_kernel(const bf16_t* __restrict__ gu,
                                                       bf16_t* __restrict__ out, int T, int I) {
  const int nvec_row = I >> 3;
  const int c = blockIdx.x * blockDim.x + threadIdx.x;  // vector within the row
  if (c >= nvec_row) return;
  for (int r = blockIdx.y; r < T; r += gridDim.y) {
    const bf16_t* g = gu + static_cast<size_t>(r) * 2 * I + c * 8;
    const u16x8 gv = *reinterpret_cast<const u16x8*>(g);
    const u16x8 uv = *reinterpret_cast<const u16x8*>(g + I);
    u16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float a = bf2f(gv[j]);
      o[j] = f2bf(__fdividef(a, 1.f + __expf(-a)) * bf2f(uv[j]));
    }
    *reinterpret_cast<u16x8*>(out + static_cast<size_t>(r) * I + c * 8) = o;
  }
}

}  // namespace

BCG_API int bcg_add_rmsnorm(const void* x, void* residual, const void* w, void* out, int T, int H,
                            float eps, int has_residual, hipStream_t stream) {
  if (H % 8 != 0 || H > NORM_THREADS * 8 * MAX_CHUNK || T <= 0) return -2;
  return launch_norm(x, residual, w, out, T, H, eps, has_residual, nullptr, stream);
}

// residual[t] <- table[tokens[t]]; out[t] <- rmsnorm(residual[t]) * w.  Token ids must be < vocab
// (checked by the caller on the host side of every path that produces them).
BCG_API int bcg_embed_rmsnorm(const int* tokens, const void* table, const void* w, void* residual, void* out,
                              int T, int H, float eps, hipStream_t stream) {
  if (H % 8 != 0 || H > NORM_THREADS * 8 * MAX_CHUNK || T <= 0) return -2;
  return launch_norm(table, residual, w, out, T, H, eps, 0, tokens, stream);
}

BCG_API int bcg_silu_mul(const void* gu, void* out, int64_t T, int I, hipStream_t stream) {
  if (I % 8 != 0 || T <= 0) return -2;
  if (T > (1 << 30) || I > (1 << 27)) return -2;
  const int bx = (I / 8 + 255) / 256;
  const int by = static_cast<int>(std::min<int64_t>(T, std::max<int64_t>(1, 8192 / bx)));
  hipLaunchKernelGGL(silu_mul_kernel, dim3(bx, by), dim3(256), 0, stream,
                     static_cast<const bf16_t*>(gu), static_cast<bf16_t*>(out), static_cast<int>(T), I);
  return BCG_CHECK_LAUNCH();
}
