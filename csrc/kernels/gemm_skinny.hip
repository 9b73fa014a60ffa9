// Projection GEMM of a few rows: C[M, N] = X[M, K] . W[N, K]^T for M <= 16, with the RMS norm of the input, the
// gated unit and the residual update fused (a decode step of one game: 4 to 16 agents).
//
// What bounds it: every weight byte is read once and meets at most 16 activation rows, so the kernel is a
// stream over W, and a CU takes in no more than about 27 GB/s, weights and activations together (measured
// over N = 4096 .. 151936, K = 896 .. 17408; all CUs: 6.2 TB/s of HBM).  Hence
//   * even shares: each of the 256 CUs owns N / 256 rows of W, in groups of 4, whatever that number is (20 rows for
//     N = 5120: blocks of 16 rows would put 320 workgroups on 256 CUs, 24.4 us where this takes 14.8); a tile of
//     the matrix instruction that the share does not fill repeats its last row, which costs no traffic;
//   * as many rows as fit share one read of X: 2 or 4 blocks of 16 rows per workgroup where N allows it;
//   * the waves of a workgroup share K, each streams its K range straight into registers, two groups of lines in
//     flight, no barrier in the loop; the partial tiles meet in LDS once, in wave order: the same inputs
//     give the same bits;
//   * one load instruction covers 8 rows x 128 bytes, whole cache lines (64-byte pieces of 16 rows, the order of the
//     matrix instruction, ran at half the rate: the vocabulary projection 484 us, this 265); a DPP rotation
//     by 8 lanes puts the halves of two loads in order;
//   * NORM: the row factor 1 / rms leaves the sum, y = rstd * sum_k (x w)[k] W[n, k]: each wave squares the
//     fragments that it loads anyway, and the factor is applied to the finished tile.  x * w is rounded to bf16
//     once, as the separate norm rounds its output once.
// 10 rows, before (norm kernel + tile GEMM with split-K, or the library) -> now, us: 7168 x 5120 24.6 -> 16.8,
// 5120 x 5120 17.6 -> 14.8, gate + up 34816 x 5120 90.6 -> 72, 151936 x 5120 277 -> 265, 18432 x 4096 79 -> 33,
// 4096 x 4096 13.4 -> 10.3, 4096 x 12288 26.1 -> 23, 896 x 896 5.8 -> 4.4, gate + up 9728 x 896 15.4 -> 8.8,
// 896 x 4864 13.1 -> 8.4; launches back to back, every one with other weights (within a captured step the profiler has 18.2, 15.4, 74
// and 265 for the first four).  Not here: M > 16 (X then takes as much of a CU's intake as W: at 20 rows 5120 x
// 5120 took 18.7 against 17.5), K > 12288 (5120 x 17408: 40 against 36.6).
#include "common.h"

namespace {

enum Epilogue { EPI_STORE = 0, EPI_SILU_MUL = 1, EPI_RESIDUAL = 2 };

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int CUS = 256;
constexpr int MAX_ROWS = 16, MAX_K = 12288;

struct SkinnyArgs {
  const uint8_t* x;        // [M, K]
  const uint8_t* w;        // [N, K]
  const bf16_t* norm_w;    // [K] (NORM)
  const bf16_t* bias;      // [N] or null
  const bf16_t* residual;  // [M, N] (EPI_RESIDUAL)
  bf16_t* c;
  int M, row_bytes, ldc, inter, units;   // units: groups of 4 output columns
  float eps, inv_k;
};

__device__ __forceinline__ float silu(float g) { return g * __builtin_amdgcn_rcpf(1.f + __expf(-g)); }

// (x * w) of 8 bf16, rounded to bf16; the squares of x are added to `ss`.
__device__ __forceinline__ bf16x8 scale_fragment(u32x4 x, u32x4 w, float& ss) {
  bf16x8 out;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float lo = __uint_as_float(x[i] << 16), hi = __uint_as_float(x[i] & 0xffff0000u);
    ss = fmaf(lo, lo, ss);
    ss = fmaf(hi, hi, ss);
    out[2 * i] = static_cast<__bf16>(lo * __uint_as_float(w[i] << 16));
    out[2 * i + 1] = static_cast<__bf16>(hi * __uint_as_float(w[i] & 0xffff0000u));
  }
  return out;
}

// Two loads cover 16 rows x 128 bytes, whole lines: `a` rows 0-7, `b` rows 8-15, lanes r and r + 8 of a
// 16-lane group the two halves of a line.  Swapping lanes r and r ^ 8 leaves the MFMA order: `a` = row r, 16-byte
// chunk kg, `b` = row r, chunk 4 + kg.
__device__ __forceinline__ void to_rows(u32x4& a, u32x4& b) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int lo = a[i], hi = b[i];
    a[i] = __builtin_amdgcn_update_dpp(lo, hi, 0x128 /*row_ror:8*/, 0xf, 0xc, false);
    b[i] = __builtin_amdgcn_update_dpp(hi, lo, 0x128, 0xf, 0x3, false);
  }
}

__device__ __forceinline__ u32x4 load_w(const uint8_t* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
}

// NW waves share K.  NT: 16-row blocks of W per workgroup (EPI_SILU_MUL: gate and up blocks of the same
// features alternate).  U: lines per group; two groups are in flight.
template <int NW, int NT, int U, int EPI, bool NORM>
__global__ __launch_bounds__(64 * NW, 4) void gemm_skinny_kernel(SkinnyArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  constexpr int PART = NT * 1024;                                // bytes of a wave's partial tile
  constexpr int BLKS = EPI == EPI_SILU_MUL ? NT / 2 : NT;        // blocks of output columns
  float* red_ss = reinterpret_cast<float*>(smem + NW * PART);    // [NW][16]
  uint8_t* norm_lds = smem + NW * PART + NW * 64;                // [row_bytes]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, kg = lane >> 4;
  // this workgroup's output columns: an even share of the groups of 4
  const int g = gridDim.x, b = blockIdx.x, q = a.units / g, rem = a.units - q * g;
  const int n0 = 4 * (b * q + min(b, rem)), cols = 4 * (q + (b < rem));

  // this wave's lines of K
  const int lines = a.row_bytes / 128;
  const int l0 = lines * wave / NW, l1 = lines * (wave + 1) / NW;

  const uint32_t chunk = (kg + (r >> 3) * 4) * 16;
  const uint8_t* wb = a.w + static_cast<size_t>(n0) * a.row_bytes;
  const uint8_t* wb_up = wb + static_cast<size_t>(a.inter) * a.row_bytes;   // EPI_SILU_MUL
  uint32_t w0[BLKS], w1[BLKS];   // rows past the share: its last row again
#pragma unroll
  for (int i = 0; i < BLKS; ++i) {
    w0[i] = static_cast<uint32_t>(min(i * 16 + (r & 7), cols - 1)) * a.row_bytes + chunk;
    w1[i] = static_cast<uint32_t>(min(i * 16 + 8 + (r & 7), cols - 1)) * a.row_bytes + chunk;
  }
  const uint32_t x0 = static_cast<uint32_t>(min(r & 7, a.M - 1)) * a.row_bytes + chunk;
  const uint32_t x1 = static_cast<uint32_t>(min(8 + (r & 7), a.M - 1)) * a.row_bytes + chunk;

  u32x4 wf[2][U][2 * NT], xf[2][U][2];
  auto load = [&](int s, int t) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t off = static_cast<uint32_t>(min(t + u, l1 - 1)) * 128;  // past the end: a line that is in cache
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        const uint8_t* base = EPI == EPI_SILU_MUL && (i & 1) ? wb_up : wb;
        const int blk = EPI == EPI_SILU_MUL ? i >> 1 : i;
        wf[s][u][2 * i] = load_w(base + off + w0[blk]);
        wf[s][u][2 * i + 1] = load_w(base + off + w1[blk]);
      }
      xf[s][u][0] = *reinterpret_cast<const u32x4*>(a.x + off + x0);
      xf[s][u][1] = *reinterpret_cast<const u32x4*>(a.x + off + x1);
    }
  };

  f32x4 acc[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float ss = 0.f;
  auto line = [&](int s, int u, int t) {
    u32x4 xa = xf[s][u][0], xb = xf[s][u][1];
    to_rows(xa, xb);
    bf16x8 x[2] = {__builtin_bit_cast(bf16x8, xa), __builtin_bit_cast(bf16x8, xb)};
    if constexpr (NORM) {
      x[0] = scale_fragment(xa, *reinterpret_cast<const u32x4*>(norm_lds + t * 128 + kg * 16), ss);
      x[1] = scale_fragment(xb, *reinterpret_cast<const u32x4*>(norm_lds + t * 128 + 64 + kg * 16), ss);
    }
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      u32x4 wa = wf[s][u][2 * i], wc = wf[s][u][2 * i + 1];
      to_rows(wa, wc);
      acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wa), x[0], acc[i], 0, 0, 0);
      acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wc), x[1], acc[i], 0, 0, 0);
    }
  };
  auto compute = [&](int s, int t) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (t + u < l1) line(s, u, t + u);
  };

  if constexpr (NORM) {  // the norm weights: the same for every row, through LDS
    for (int i = threadIdx.x * 16; i < a.row_bytes; i += 64 * NW * 16)
      *reinterpret_cast<u32x4*>(norm_lds + i) = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint8_t*>(a.norm_w) + i);
  }
  if (l0 < l1) load(0, l0);
  if constexpr (NORM) __syncthreads();
  for (int t = l0; t < l1; t += 2 * U) {
    load(1, t + U);
    compute(0, t);
    load(0, t + 2 * U);
    compute(1, t + U);
  }

  // the waves' partial tiles and squares, summed in wave order
#pragma unroll
  for (int i = 0; i < NT; ++i) *reinterpret_cast<f32x4*>(smem + wave * PART + i * 1024 + lane * 16) = acc[i];
  if constexpr (NORM) {
    ss += __shfl_xor(ss, 16);
    ss += __shfl_xor(ss, 32);
    if (lane < 16) red_ss[wave * 16 + lane] = ss;
  }
  __syncthreads();

  // lane holds D[n = 4 kg + e][m = r] of a block
  const int i = wave, n = n0 + i * 16 + 4 * kg;
  if (i >= BLKS || r >= a.M || i * 16 + 4 * kg >= cols) return;
  auto total = [&](int blk) {
    f32x4 v = *reinterpret_cast<const f32x4*>(smem + blk * 1024 + lane * 16);
#pragma unroll
    for (int w = 1; w < NW; ++w) v += *reinterpret_cast<const f32x4*>(smem + w * PART + blk * 1024 + lane * 16);
    return v;
  };
  float rs = 1.f;
  if constexpr (NORM) {
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) s += red_ss[w * 16 + r];
    rs = rsqrtf(s * a.inv_k + a.eps);
  }
  f32x4 v;
  if constexpr (EPI == EPI_SILU_MUL) {
    const f32x4 gate = total(2 * i) * rs, up = total(2 * i + 1) * rs;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = silu(gate[e]) * up[e];
  } else {
    v = total(i) * rs;
    if (a.bias != nullptr) {
      const u16x4 bb = *reinterpret_cast<const u16x4*>(a.bias + n);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += bf2f(bb[e]);
    }
    if constexpr (EPI == EPI_RESIDUAL) {
      const u16x4 rr = *reinterpret_cast<const u16x4*>(a.residual + static_cast<size_t>(r) * a.ldc + n);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += bf2f(rr[e]);
    }
  }
  u16x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = f2bf(v[e]);
  *reinterpret_cast<u16x4*>(a.c + static_cast<size_t>(r) * a.ldc + n) = o;
}

template <int NW, int NT, int U, int EPI, bool NORM>
int launch(const SkinnyArgs& a, hipStream_t stream) {
  constexpr int MOST = EPI == EPI_SILU_MUL ? 2 * NT : 4 * NT;        // groups of 4 columns that a workgroup can hold
  const int passes = (a.units + CUS * MOST - 1) / (CUS * MOST);      // workgroups per CU
  const int grid = a.units < CUS * passes ? a.units : CUS * passes;
  const int lds = NW * (NT * 1024 + 64) + (NORM ? a.row_bytes : 0);
  hipLaunchKernelGGL((gemm_skinny_kernel<NW, NT, U, EPI, NORM>), dim3(grid), dim3(64 * NW), lds, stream, a);
  return BCG_CHECK_LAUNCH();
}

// The fewest row blocks that hold a CU's share in one workgroup, 4 at most: blocks that stay empty cost matrix
// instructions (4096 x 4096: 1 block 10.3 us, 2 blocks 12.3), fewer than the share fills cost reads of X
// (10240 x 5120: 2 blocks 29.4, 4 blocks 26.6).  4 waves where a wave's K range would be short
// (896 x 4864: 8.4 us against 9.7 with 8), 8 to keep enough lines in flight otherwise (4096 x 12288: 23.0, 24.4).
template <int EPI, bool NORM>
int pick(const SkinnyArgs& a, hipStream_t s) {
  const int share = (a.units + CUS - 1) / CUS;
  if constexpr (EPI == EPI_SILU_MUL) {
    return share <= 4 ? launch<8, 2, 1, EPI, NORM>(a, s) : launch<8, 4, 1, EPI, NORM>(a, s);
  } else {
    if (share <= 4) return a.row_bytes < 16384 ? launch<4, 1, 2, EPI, NORM>(a, s) : launch<8, 1, 2, EPI, NORM>(a, s);
    return share <= 8 ? launch<8, 2, 1, EPI, NORM>(a, s) : launch<8, 4, 1, EPI, NORM>(a, s);
  }
}

}  // namespace

// epi: 0 = store (+bias), 1 = silu(gate)*up into [M, N / 2], 2 = residual + acc (+bias).  norm_w: RMS-normalise the rows
// of x with these weights first (epi 0, 1).  1 <= M <= 16, K % 64 == 0, 64 <= K <= 12288, the output width a multiple
// of 4; rows contiguous, x and w 16-byte aligned, the others 8-byte aligned.
BCG_API int bcg_gemm_skinny(int epi, const void* x, const void* w, const void* norm_w, float eps, const void* bias,
                            const void* residual, void* c, int M, int N, int K, hipStream_t stream) {
  const int n_out = epi == EPI_SILU_MUL ? N / 2 : N;
  if (M < 1 || M > MAX_ROWS || K < 64 || K > MAX_K || K % 64 || n_out < 4 || n_out % 4 || (epi == EPI_SILU_MUL && N % 2)) return -2;
  const SkinnyArgs a{static_cast<const uint8_t*>(x), static_cast<const uint8_t*>(w), static_cast<const bf16_t*>(norm_w),
                     static_cast<const bf16_t*>(bias), static_cast<const bf16_t*>(residual), static_cast<bf16_t*>(c),
                     M, 2 * K, n_out, N / 2, n_out / 4, eps, 1.f / K};
  switch (epi) {
    case EPI_STORE: return norm_w ? pick<EPI_STORE, true>(a, stream) : pick<EPI_STORE, false>(a, stream);
    case EPI_SILU_MUL:
      if (bias) return -2;
      return norm_w ? pick<EPI_SILU_MUL, true>(a, stream) : pick<EPI_SILU_MUL, false>(a, stream);
    case EPI_RESIDUAL:
      if (!residual || norm_w) return -2;
      return pick<EPI_RESIDUAL, false>(a, stream);
    default: return -2;
  }
}
