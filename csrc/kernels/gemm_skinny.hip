// Projection GEMM of a few rows: C[M, N] = X[M, K] . W[N, K]^T for M <= 64 in bf16, <= 32 in fp8 (e4m3, row and column scales), with
// the RMS norm of the input, the gated unit and the residual update fused (a decode step of one to three games).
//
// What bounds it: every weight byte is read once and meets a few dozen activation rows at most, so the kernel is a stream over W.  Plain
// streaming loads of such weights reach 6.7 TB/s at 356 MB and 6.1 at 84 MB, launch included; the rest is what a CU takes in:
// X comes from L2 once per CU, and a CU's load path follows the address quads: four neighbouring lanes that read 64 bytes of
// one row cost a quarter of four that read 16 bytes of four rows (the order of the matrix instruction): 117 and 36 B/ns per CU
// out of L2.  Hence
//   * even shares: each of the 256 CUs owns N / 256 rows of W, in groups of 4, whatever that number is (blocks of 16 rows would
//     put 320 workgroups on 256 CUs for N = 5120), as one workgroup that streams its rows pass after pass (up to 8 blocks of 16
//     rows at once): the next pass's loads are in flight while a pass is reduced and written (34816 x 5120 gated, 10 rows:
//     three workgroups per CU, one after the other, 74 us, so 59; 151936 x 5120 265 -> 234);
//   * the waves of a workgroup share K in turns, unit by unit: neighbouring waves read neighbouring lines (4 % over
//     a contiguous part of K per wave).  Rows of 8 and 16 KB may be shared in contiguous parts (`meets_channels`): in turns, all
//     waves of the chip read the same few memory channels at a time (1 to 10 rows, us, in turns and in parts: 8192 x 8192 30.2, 25.5;
//     4096 x 8192 16.5, 13.5; 8192 x 4096 15.9, 15.2; 4096 x 4096 8.8, 8.0; but rows of 32 KB, 8192 x 16384 58, 83).  Rows of
//     32 KB are shared in turns, a workgroup beginning at its own (4096 x 16384 33.5, so 25.5, library 31.3; but 16384 x 4096
//     25.7, 31).  No barrier in the loop, every register is loaded again as soon as it has been consumed; the partial tiles meet in LDS once per pass, in wave order: the same inputs give the same bits;
//   * a unit of K is 256 bytes: a load takes 64 bytes of each of 16 (row, segment) pairs, and a 4 x 4 transposition within
//     quads of lanes makes the operands of four matrix instructions (5120 x 17408 with 10 rows 36.2 -> 31.9 us, fp8 6144 x 16384
//     with 20 rows 25.2 -> 20.8).  Short rows and shares of 4 columns use units of 128 bytes, 8 rows a load and one rotation by 8
//     lanes (9728 x 896 gated 8.1 -> 7.3, 896 x 4864 8.6 -> 7.7): with 7 units of 256 bytes a wave has nothing to overlap;
//   * rows past the share, past M and past K lie outside the buffer descriptors: they read as zeros without traffic;
//   * NORM: the row factor 1 / rms leaves the sum, y = rstd * sum_k (x w)[k] W[n, k]: each wave squares the
//     fragments that it loads anyway, and the factor is applied to the finished tile.  x * w is rounded to bf16
//     once, as the separate norm rounds its output once.
// 10 rows, us, one workgroup per pass and 128-byte units -> now: 7168 x 5120 18.1 -> 16.4, 5120 x 5120 14.7 -> 12.4, gate + up 34816 x
// 5120 74.5 -> 59.8, 151936 x 5120 265 -> 234, 4096 x 4096 10.3 -> 9.2, 4096 x 12288 23 -> 18.7, 5120 x 17408 (tile kernel 36.6) 31.9.
// 1 row, against the same: 2048 x 8192 10.6 -> 10.3, but up to 1024 x 8192 9.3 -> 9.8, 1024 x 12288 12.4 -> 13.6.
// 20 rows, tile kernel with split-K -> now: fp8 8192 x 6144 15.4 -> 11.6, 6144 x 6144 14.8 -> 10.5, 32768 x 6144 38.5 -> 35.1, 6144 x
// 16384 27.4 -> 20.8; bf16 32768 x 6144 75.4 -> 68.6.  Launches in a graph, every one with other weights.  From 33 rows on X takes
// more of a CU's intake than W, and two blocks of W fill the registers: short rows in one pass only (64 rows, library -> here:
// 4096 x 2048 12.4 -> 9.5; 4096 x 4096: tile kernel 13.8, here 14.9).
#include <type_traits>

#include "common.h"

namespace {

enum Epilogue { EPI_STORE = 0, EPI_SILU_MUL = 1, EPI_RESIDUAL = 2 };

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef int i32x8 __attribute__((ext_vector_type(8)));

constexpr int CUS = 256, NW = 8;             // workgroups, waves of one
constexpr int MAX_ROWS = 64, MAX_NORM_ROWS = 16, MAX_ROW_BYTES = 65536, MAX_NORM_K = 16384;
constexpr uint32_t PAST_END = 0x80000000u;   // an offset outside every descriptor
constexpr int ROUND_KB = 64;                 // LDS of one round of a reduction

struct SkinnyArgs {
  const uint8_t* x;        // [M, K]
  const uint8_t* w;        // [N, K]
  const bf16_t* norm_w;    // [K] (NORM)
  const bf16_t* bias;      // [N] or null
  const bf16_t* residual;  // [M, N] (EPI_RESIDUAL)
  bf16_t* c;
  const float* x_scale;    // [M], [N] (F8)
  const float* w_scale;
  int M, row_bytes, ldc, inter, units, passes;   // units: groups of 4 output columns
  float eps, inv_k;
};

__device__ __forceinline__ float silu(float g) { return g * __builtin_amdgcn_rcpf(1.f + __expf(-g)); }

// (x * w) of 8 bf16, rounded to bf16; the squares of x are added to `ss`.
__device__ __forceinline__ u32x4 scale_fragment(u32x4 x, u32x4 w, float& ss) {
  bf16x8 out;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float lo = __uint_as_float(x[i] << 16), hi = __uint_as_float(x[i] & 0xffff0000u);
    ss = fmaf(lo, lo, ss);
    ss = fmaf(hi, hi, ss);
    out[2 * i] = static_cast<__bf16>(lo * __uint_as_float(w[i] << 16));
    out[2 * i + 1] = static_cast<__bf16>(hi * __uint_as_float(w[i] & 0xffff0000u));
  }
  return __builtin_bit_cast(u32x4, out);
}

// 256-byte units.  Load i of a block takes rows 4 g + i (g = lane bits 2, 3), lane bits 4, 5 the 64-byte segment, the quad
// its four 16-byte chunks; transposed within quads lane q holds row 4 g + q = lane & 15, out[j] chunk j.
__device__ __forceinline__ void to_operand(const u32x4 (&in)[4], u32x4 (&out)[4]) { quad_transpose(in, out); }

// 128-byte units.  The two loads of a block cover 16 rows x 128 bytes: in[0] rows 0-7, in[1] rows 8-15, lanes r and r + 8 of a
// 16-lane group the two halves of a line.  Swapping lanes r and r ^ 8: out[0] = row r, chunk kg, out[1] = row r, chunk 4 + kg.
__device__ __forceinline__ void to_operand(const u32x4 (&in)[2], u32x4 (&out)[2]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int lo = in[0][i], hi = in[1][i];
    out[0][i] = __builtin_amdgcn_update_dpp(lo, hi, 0x128 /*row_ror:8*/, 0xf, 0xc, false);
    out[1][i] = __builtin_amdgcn_update_dpp(hi, lo, 0x128, 0xf, 0x3, false);
  }
}

__device__ __forceinline__ i32x8 join(u32x4 a, u32x4 b) {
  return i32x8{static_cast<int>(a[0]), static_cast<int>(a[1]), static_cast<int>(a[2]), static_cast<int>(a[3]),
               static_cast<int>(b[0]), static_cast<int>(b[1]), static_cast<int>(b[2]), static_cast<int>(b[3])};
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}

template <int MT, int NT, int EPI>
struct Reduction {   // of a pass's partial tiles, OB output blocks at a time
  static constexpr int PAIR = EPI == EPI_SILU_MUL ? 2 : 1;          // accumulators of an output block
  static constexpr int OUT = NT / PAIR * MT;                        // output blocks of 16 x 16
  static constexpr int ROUNDS = (NW * OUT * PAIR + ROUND_KB - 1) / ROUND_KB;
  static constexpr int OB = (OUT + ROUNDS - 1) / ROUNDS;
  static constexpr int PART = OB * PAIR * 1024;                     // bytes of a wave's share of a round
  static constexpr int LDS = NW * (PART + MT * 64);
};

// MT, NT: blocks of 16 rows of X and of W (EPI_SILU_MUL: gate and up blocks of the same features alternate).  UB: bytes of
// a unit of K.  D: units in flight per wave.  ORD: the orders of `meets_channels` (instances of their own: their index arithmetic costs
// 0.8 % of a step of small launches).
template <int MT, int NT, int UB, int D, int EPI, bool NORM, bool F8, bool ORD>
__global__ __launch_bounds__(64 * NW, 2) void gemm_skinny_kernel(SkinnyArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  using Red = Reduction<MT, NT, EPI>;
  constexpr int LB = UB / 64;                                       // loads of a block and unit
  constexpr int PAIR = Red::PAIR, OUT = Red::OUT, OB = Red::OB, PART = Red::PART;
  float* red_ss = reinterpret_cast<float*>(smem + NW * PART);       // [NW][MT][16]
  uint8_t* norm_lds = smem + Red::LDS;                              // [lw * NW * UB], zeros past K
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, kg = lane >> 4;
  // this workgroup's output columns: an even share of the groups of 4, `per` of them a pass
  const int g = gridDim.x, b = blockIdx.x, q = a.units / g, rem = a.units - q * g;
  const int n0 = 4 * (b * q + min(b, rem)), share = 4 * (q + (b < rem));
  const int per = (share / 4 + a.passes - 1) / a.passes * 4;
  const uint32_t rb = a.row_bytes;
  const int nu = (rb + UB - 1) / UB, lw = (nu + NW - 1) / NW;       // units of K, a wave's units of a pass
  auto unit = [&](int j) {                                          // of K, the j-th of this wave
    if constexpr (!ORD) return wave + j * NW;
    if (rb != 32768) return wave * lw + j;
    j += static_cast<int>(blockIdx.x >> 3) % lw;
    return wave + (j < lw ? j : j - lw) * NW;
  };
  const uint32_t vo = UB == 256 ? ((lane >> 2) & 3) * 4 * rb + kg * 64 + (lane & 3) * 16 : (r & 7) * rb + (kg + (r >> 3) * 4) * 16;
  const uint32_t vs = UB == 256 ? rb : 8 * rb;                      // from load to load of a block
  const uint32_t vo_tail = UB == 256 && (rb & 255) && kg >= 2 ? PAST_END : vo;   // the last unit may be half a unit
  const uint8_t* wb = a.w + static_cast<size_t>(n0) * rb;
  const uint8_t* wb_up = wb + static_cast<size_t>(a.inter) * rb;    // EPI_SILU_MUL

  u32x4 wf[D][NT][LB], xf[D][MT][LB];
  struct Item {
    int p, j;   // pass, unit of this wave
  };
  struct Where {
    const uint8_t *w, *up, *x;
    int w_bytes, x_bytes;   // from the unit's first byte to the end of the pass's rows (of X)
    bool tail;
  };
  auto advance = [&](Item& it) {
    if (++it.j == lw) {
      it.j = 0;
      ++it.p;
    }
  };
  auto where = [&](Item it) {
    const int t = unit(it.j);
    const bool in = t < nu && it.p < a.passes;
    const int off = in ? t * UB : 0, first = in ? it.p * per : 0;
    const size_t at = static_cast<size_t>(first) * rb + off;
    return Where{wb + at, wb_up + at, a.x + off, in ? min(per, share - first) * static_cast<int>(rb) - off : 0,
                 in ? a.M * static_cast<int>(rb) - off : 0, in && t + 1 == nu};
  };
  auto fetch = [&](const uint8_t* base, int bytes, int blk, bool tail, auto aux, u32x4 (&out)[LB]) {
    const int skip = blk * 16 * static_cast<int>(rb);
    const __amdgpu_buffer_rsrc_t rs = rsrc(base + skip, max(bytes - skip, 0));
    const uint32_t v = tail ? vo_tail : vo;
#pragma unroll
    for (int i = 0; i < LB; ++i) out[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, v + i * vs, 0, decltype(aux)::value);
  };
  using Kept = std::integral_constant<int, 0>;
  using Streamed = std::integral_constant<int, 2>;   // nt: read once
  auto load_x = [&](const Where& at, int s, int m) { fetch(at.x, at.x_bytes, m, at.tail, Kept{}, xf[s][m]); };
  auto load_w = [&](const Where& at, int s, int n) {
    fetch(PAIR == 2 && (n & 1) ? at.up : at.w, at.w_bytes, n / PAIR, at.tail, Streamed{}, wf[s][n]);
  };

  f32x4 acc[NT][MT];
  float ss[MT];
  auto clear = [&] {
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < MT; ++j) ss[j] = 0.f;
  };

  // output block `ob` of a pass: lane holds D[n = 4 kg + e][m = r]
  auto write_out = [&](int p, int ob, f32x4 v, f32x4 up) {
    const int i = ob / MT, j = ob % MT, m = j * 16 + r, c = i * 16 + 4 * kg, n = n0 + p * per + c;
    if (m >= a.M || c >= min(per, share - p * per)) return;
    if constexpr (NORM) {
      float s = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) s += red_ss[(w * MT + j) * 16 + r];
      const float rs = rsqrtf(s * a.inv_k + a.eps);
      v *= rs;
      up *= rs;
    }
    if constexpr (EPI == EPI_SILU_MUL) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = silu(v[e]) * up[e];
    } else {
      if constexpr (F8) {
        const float xs = a.x_scale[m];
        const f32x4 wsc = *reinterpret_cast<const f32x4*>(a.w_scale + n);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] *= xs * wsc[e];
      }
      if (a.bias != nullptr) {
        const u16x4 bb = *reinterpret_cast<const u16x4*>(a.bias + n);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += bf2f(bb[e]);
      }
      if constexpr (EPI == EPI_RESIDUAL) {
        const u16x4 rr = *reinterpret_cast<const u16x4*>(a.residual + static_cast<size_t>(m) * a.ldc + n);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += bf2f(rr[e]);
      }
    }
    u16x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = f2bf(v[e]);
    *reinterpret_cast<u16x4*>(a.c + static_cast<size_t>(m) * a.ldc + n) = o;
  };

  // the waves' partial tiles and squares, summed in wave order; loads of the next pass stay in flight
  auto finish = [&](int p) {
    if constexpr (NORM) {
#pragma unroll
      for (int j = 0; j < MT; ++j) {
        ss[j] += __shfl_xor(ss[j], 16);
        ss[j] += __shfl_xor(ss[j], 32);
        if (lane < 16) red_ss[(wave * MT + j) * 16 + lane] = ss[j];
      }
    }
#pragma unroll
    for (int rd = 0; rd < Red::ROUNDS; ++rd) {
#pragma unroll
      for (int o = 0; o < OB; ++o) {
        const int ob = rd * OB + o;
        if (ob >= OUT) break;
#pragma unroll
        for (int h = 0; h < PAIR; ++h)
          *reinterpret_cast<f32x4*>(smem + wave * PART + (o * PAIR + h) * 1024 + lane * 16) = acc[ob / MT * PAIR + h][ob % MT];
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      auto total = [&](int blk) {
        f32x4 v = *reinterpret_cast<const f32x4*>(smem + blk * 1024 + lane * 16);
#pragma unroll
        for (int w = 1; w < NW; ++w) v += *reinterpret_cast<const f32x4*>(smem + w * PART + blk * 1024 + lane * 16);
        return v;
      };
      for (int o = wave; o < OB; o += NW)
        if (rd * OB + o < OUT) write_out(p, rd * OB + o, total(PAIR * o), PAIR == 2 ? total(PAIR * o + PAIR - 1) : f32x4{});
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();   // before the next round's partial tiles
    }
  };

  constexpr int NV = 2;   // 16-byte pieces of the norm weights per thread that are asked for before the first units
  u32x4 nv[NV];
  if constexpr (NORM) {
#pragma unroll
    for (int i = 0; i < NV; ++i)
      nv[i] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint8_t*>(a.norm_w) + min((threadIdx.x + i * 64 * NW) * 16, rb - 16));
  }
  Item now{0, 0}, next{0, 0};   // the unit at hand, the next one to load
#pragma unroll
  for (int s = 0; s < D; ++s) {
    const Where at = where(next);
    advance(next);
#pragma unroll
    for (int m = 0; m < MT; ++m) load_x(at, s, m);
#pragma unroll
    for (int n = 0; n < NT; ++n) load_w(at, s, n);
  }
  if constexpr (NORM) {   // the norm weights: the same for every row, through LDS
    const uint32_t end = static_cast<uint32_t>(lw) * NW * UB;
    for (uint32_t i = threadIdx.x * 16, k = 0; i < end; i += 64 * NW * 16, ++k) {
      u32x4 v = {0, 0, 0, 0};
      if (i < rb) v = k == 0 ? nv[0] : k == 1 ? nv[1] : *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint8_t*>(a.norm_w) + i);
      *reinterpret_cast<u32x4*>(norm_lds + i) = v;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
  }
  clear();
  while (true) {
#pragma unroll
    for (int s = 0; s < D; ++s) {
      const Where at = where(next);
      advance(next);
      u32x4 xt[MT][LB];
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        to_operand(xf[s][m], xt[m]);
        load_x(at, s, m);
        if constexpr (NORM) {
          const uint8_t* nw = norm_lds + unit(now.j) * UB;
#pragma unroll
          for (int j = 0; j < LB; ++j)
            xt[m][j] = scale_fragment(xt[m][j], *reinterpret_cast<const u32x4*>(nw + (UB == 256 ? kg * 64 + j * 16 : j * 64 + kg * 16)), ss[m]);
        }
        __builtin_amdgcn_sched_barrier(0);   // a register is loaded again where it was consumed, not later
      }
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        u32x4 wt[LB];
        to_operand(wf[s][n], wt);
        load_w(at, s, n);
        if constexpr (F8) {   // 32 bytes of a row an operand; formats 0 / 0 = e4m3, scales 127 = 1
#pragma unroll
          for (int j = 0; j < LB; j += 2)
#pragma unroll
            for (int m = 0; m < MT; ++m)
              acc[n][m] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(join(wt[j], wt[j + 1]), join(xt[m][j], xt[m][j + 1]),
                                                                            acc[n][m], 0, 0, 0, 127, 0, 127);
        } else {
#pragma unroll
          for (int j = 0; j < LB; ++j)
#pragma unroll
            for (int m = 0; m < MT; ++m)
              acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wt[j]), __builtin_bit_cast(bf16x8, xt[m][j]),
                                                                   acc[n][m], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (now.j + 1 == lw) {
        finish(now.p);
        if (now.p + 1 == a.passes) return;
        clear();
      }
      advance(now);
    }
  }
}

// Whether the workgroups meet in the same memory channels if all begin at the same unit of K: many rows of 32 KB, and of 8 and 16 KB where the
// shares are 2^n bytes apart (one part of K per wave instead of turns: 4096 and 8192 rows 0.84 to 0.97 of the time, but fp8 5120 and 6144 x 8192
// 1.02 to 1.05, 6144 x 16384 0.96 to 1.01).
bool meets_channels(const SkinnyArgs& a) {
  if (a.row_bytes == 32768) return a.units >= 2 * CUS;   // (1024 x 16384: 16.6, so 17.9)
  const int64_t share = static_cast<int64_t>(a.units / CUS) * 4 * a.row_bytes;
  return (a.row_bytes == 8192 || a.row_bytes == 16384) && a.units % CUS == 0 && share >= 131072 && (share & (share - 1)) == 0;
}

template <int MT, int NT, int UB, int D, int EPI, bool NORM, bool F8>
int launch(SkinnyArgs a, int passes, hipStream_t stream) {
  a.passes = passes;
  const int nu = (a.row_bytes + UB - 1) / UB;
  const int lds = Reduction<MT, NT, EPI>::LDS + (NORM ? (nu + NW - 1) / NW * NW * UB : 0);
  auto kernel = gemm_skinny_kernel<MT, NT, UB, D, EPI, NORM, F8, false>;
  if constexpr (UB == 256 || D == 2)   // (the others are for shorter rows)
    if (meets_channels(a)) kernel = gemm_skinny_kernel<MT, NT, UB, D, EPI, NORM, F8, true>;
  if (lds > 65536 && hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
    return -1;
  hipLaunchKernelGGL(kernel, dim3(a.units < CUS ? a.units : CUS), dim3(64 * NW), lds, stream, a);
  return BCG_CHECK_LAUNCH();
}

// The fewest passes, then the fewest row blocks that hold a pass: blocks that stay empty cost instructions.  Rows of up to
// 2048 bytes and shares of 4 columns take 128-byte units (see above), the latter two units at once: a wave then has only
// four loads in flight (896 x 4864: 8.5 us with one, 7.7); up to four rows, whose loads of X are mostly outside, shares of
// 8 columns too (2048 x 8192: 11.6, 10.3).
template <int MT, int EPI, bool NORM, bool F8>
int pick(const SkinnyArgs& a, hipStream_t s) {
  constexpr int PER = EPI == EPI_SILU_MUL ? 2 : 4;                             // groups of 4 columns of a block of W
  constexpr int MOST = MT >= 3 ? 2 : MT == 2 ? 4 : EPI == EPI_SILU_MUL ? 6 : 8;   // (registers of two waves per SIMD)
  const int share = (a.units + CUS - 1) / CUS, passes = (share + MOST * PER - 1) / (MOST * PER);
  const int blocks = ((share + passes - 1) / passes + PER - 1) / PER;
  if constexpr (MT == 1 && !F8) {
    if (a.row_bytes <= 2048) {
      if constexpr (EPI == EPI_SILU_MUL) {
        return blocks <= 2 ? launch<1, 2, 128, 1, EPI, NORM, F8>(a, passes, s)
                           : blocks <= 4 ? launch<1, 4, 128, 1, EPI, NORM, F8>(a, passes, s) : launch<1, 6, 128, 1, EPI, NORM, F8>(a, passes, s);
      } else {
        return blocks <= 1   ? launch<1, 1, 128, 1, EPI, NORM, F8>(a, passes, s)
               : blocks <= 2 ? launch<1, 2, 128, 1, EPI, NORM, F8>(a, passes, s)
               : blocks <= 4 ? launch<1, 4, 128, 1, EPI, NORM, F8>(a, passes, s) : launch<1, 8, 128, 1, EPI, NORM, F8>(a, passes, s);
      }
    }
    if (share == 1 || (EPI != EPI_SILU_MUL && share == 2 && a.M <= 4)) return launch<1, EPI == EPI_SILU_MUL ? 2 : 1, 128, 2, EPI, NORM, F8>(a, passes, s);
  }
  if constexpr (EPI == EPI_SILU_MUL) {
    if (blocks <= 2) return launch<MT, 2, 256, 1, EPI, NORM, F8>(a, passes, s);
    if constexpr (MT == 1)
      if (blocks > 4) return launch<MT, 6, 256, 1, EPI, NORM, F8>(a, passes, s);
    if constexpr (MT <= 2) return launch<MT, 4, 256, 1, EPI, NORM, F8>(a, passes, s);
    return -2;
  } else {
    if (blocks <= 1) return launch<MT, 1, 256, 1, EPI, NORM, F8>(a, passes, s);
    if (blocks <= 2) return launch<MT, 2, 256, 1, EPI, NORM, F8>(a, passes, s);
    if constexpr (MT == 1)
      if (blocks > 4) return launch<MT, 8, 256, 1, EPI, NORM, F8>(a, passes, s);
    if constexpr (MT <= 2) return launch<MT, 4, 256, 1, EPI, NORM, F8>(a, passes, s);
    return -2;
  }
}

// by the blocks of 16 rows
template <int EPI, bool F8>
int pick_rows(const SkinnyArgs& a, hipStream_t s) {
  if (a.M <= 16) return pick<1, EPI, false, F8>(a, s);
  if (a.M <= 32) return pick<2, EPI, false, F8>(a, s);
  if constexpr (!F8) return a.M <= 48 ? pick<3, EPI, false, false>(a, s) : pick<4, EPI, false, false>(a, s);
  return -2;
}

bool covered(int M, int row_bytes, int n_out) {
  return M >= 1 && M <= MAX_ROWS && row_bytes >= 128 && row_bytes <= MAX_ROW_BYTES && row_bytes % 128 == 0 && n_out >= 4 && n_out % 4 == 0;
}

}  // namespace

// epi: 0 = store (+bias), 1 = silu(gate)*up into [M, N / 2], 2 = residual + acc (+bias).  norm_w: RMS-normalise the rows
// of x with these weights first (epi 0, 1; M <= 16, K <= 16384).  1 <= M <= 64, K % 64 == 0, 64 <= K <= 32768, the output
// width a multiple of 4; rows contiguous, x and w 16-byte aligned, the others 8-byte aligned.
BCG_API int bcg_gemm_skinny(int epi, const void* x, const void* w, const void* norm_w, float eps, const void* bias,
                            const void* residual, void* c, int M, int N, int K, hipStream_t stream) {
  const int n_out = epi == EPI_SILU_MUL ? N / 2 : N;
  if (K < 1 || K > MAX_ROW_BYTES / 2 || !covered(M, 2 * K, n_out) || (epi == EPI_SILU_MUL && N % 2)) return -2;
  if (norm_w && (M > MAX_NORM_ROWS || K > MAX_NORM_K)) return -2;
  const SkinnyArgs a{static_cast<const uint8_t*>(x), static_cast<const uint8_t*>(w), static_cast<const bf16_t*>(norm_w),
                     static_cast<const bf16_t*>(bias), static_cast<const bf16_t*>(residual), static_cast<bf16_t*>(c), nullptr, nullptr,
                     M, 2 * K, n_out, N / 2, n_out / 4, 1, eps, 1.f / K};
  switch (epi) {
    case EPI_STORE:
      if (norm_w) return pick<1, EPI_STORE, true, false>(a, stream);
      return pick_rows<EPI_STORE, false>(a, stream);
    case EPI_SILU_MUL:
      if (bias) return -2;
      if (norm_w) return pick<1, EPI_SILU_MUL, true, false>(a, stream);
      return pick_rows<EPI_SILU_MUL, false>(a, stream);
    case EPI_RESIDUAL:
      if (!residual || norm_w) return -2;
      return pick_rows<EPI_RESIDUAL, false>(a, stream);
    default: return -2;
  }
}

// fp8 (e4m3fn) form: C = x_scale[m] * w_scale[n] * (Xq . Wq^T) (+ bias) (+ residual); epi 0 or 2.  1 <= M <= 32, K % 128 == 0,
// K <= 65536, N a multiple of 4; rows contiguous, xq, wq and w_scale 16-byte aligned, the others 8-byte aligned.
BCG_API int bcg_gemm_skinny_fp8(int epi, const void* xq, const void* wq, const float* x_scale, const float* w_scale, const void* bias,
                                const void* residual, void* c, int M, int N, int K, hipStream_t stream) {
  if (!covered(M, K, N) || M > 32 || !x_scale || !w_scale) return -2;
  const SkinnyArgs a{static_cast<const uint8_t*>(xq), static_cast<const uint8_t*>(wq), nullptr, static_cast<const bf16_t*>(bias),
                     static_cast<const bf16_t*>(residual), static_cast<bf16_t*>(c), x_scale, w_scale,
                     M, K, N, 0, N / 4, 1, 0.f, 0.f};
  switch (epi) {
    case EPI_STORE: return pick_rows<EPI_STORE, true>(a, stream);
    case EPI_RESIDUAL:
      if (!residual) return -2;
      return pick_rows<EPI_RESIDUAL, true>(a, stream);
    default: return -2;
  }
}
