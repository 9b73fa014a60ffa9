// Per-head products of the latent mixers, bf16: out[t, h] = x[t, h] w[h], w [H, K, N] as it lies, with what stands around them:
// the turned tail of the queries (`tail`), or the sigmoid gate on the result (`gate`).
//
// One workgroup per (64 to 512 tokens, head, 64 or 128 columns), four waves of 16 tokens.  The head's weight columns are turned into LDS once
// ([column][input]: a lane's operand is 16 bytes of one column), the tokens' rows come straight from memory, 16 bytes per lane, those of
// the next 64 tokens under the products of these; products are W^T X^T, so that a lane holds neighbouring columns of one token.
// Bound by memory in large steps (8 bytes per product of 128: below the matrix rate by ten), by the launch in small ones.  Measured beside the
// vendor's batched product and the kernels of the tail and the gate (heads of 128 -> 128, tails of 64), us in a captured graph: queries with their
// tail, 64 tokens, 16 heads 7.2 -> 3.5; 2039, 16 14.6 -> 7.8; 8183, 32 56 -> 41 (4.9 TB/s); results with their gate 7.2 -> 5.1, 16.9 -> 11.5, 79 -> 52; products
// alone 5.1 -> 3.4, 7.4 -> 7.2, 36 -> 31.
#include <algorithm>

#include "seqmix_common.h"

namespace {

constexpr int NT = 256;
typedef short s16x8 __attribute__((ext_vector_type(8)));   // bits of eight bf16

struct HeadArgs {
  const bf16_t* x; int64_t x_row, x_head;
  const bf16_t* w;                                   // [H, K, N]
  bf16_t* out; int64_t o_row, o_head;
  int T, H, N, tiles;                                // tiles: of 64 tokens, per workgroup
  // the tail: x[t, h, K ..] turned (as rope_tail_kernel does) into out[t, h, N ..]; n 0: none
  const int* positions; const float* inv_freq; int n, half, pairs; float amp;
  // sigmoid gate on the rounded result (null: none); one gate column for `group` columns of [H, N]
  const bf16_t* gate; int64_t gate_row; int group;
};

__device__ __forceinline__ float sigmoid(float z) { return 1.0f / (1.0f + expf(-z)); }

// The tails of tokens t_first .. t_end - 1 and heads h0 .. h1 - 1: a thread takes one token's sines once for all of them, V
// neighbouring pairs where the halves allow it.
template <int V>
__device__ __forceinline__ void turn_tails(const HeadArgs& a, int K, int t_first, int t_end, int h0, int h1) {
  const bool vec = !a.pairs && a.n == 2 * a.half && a.half % 8 == 0;
  typedef short Bits __attribute__((ext_vector_type(V)));
  const int per = vec ? a.half / V : a.n - a.half;   // items of a token: V pairs each, or pairs and then copied features
  for (int e = threadIdx.x; e < (t_end - t_first) * per; e += NT) {
    const int t = t_first + e / per, j = e % per;
    const bf16_t* src = a.x + t * a.x_row + h0 * a.x_head + K;
    bf16_t* dst = a.out + t * a.o_row + h0 * a.o_head + a.N;
    const float pos = static_cast<float>(a.positions[t]);
    float cs[V] = {}, sn[V] = {};
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const int f = vec ? V * j + i : j;
      if (f < a.half && (vec || i == 0)) sincosf(pos * a.inv_freq[f], &sn[i], &cs[i]);
      sn[i] *= a.amp;
      cs[i] *= a.amp;
    }
    for (int h = h0; h < h1; ++h, src += a.x_head, dst += a.o_head) {
      if (vec) {
        const Bits u = *reinterpret_cast<const Bits*>(src + V * j), v = *reinterpret_cast<const Bits*>(src + a.half + V * j);
        Bits p, q;
#pragma unroll
        for (int i = 0; i < V; ++i) {
          const float uf = bf2f(static_cast<bf16_t>(u[i])), vf = bf2f(static_cast<bf16_t>(v[i]));
          p[i] = static_cast<short>(f2bf(uf * cs[i] - vf * sn[i]));
          q[i] = static_cast<short>(f2bf(vf * cs[i] + uf * sn[i]));
        }
        *reinterpret_cast<Bits*>(dst + V * j) = p;
        *reinterpret_cast<Bits*>(dst + a.half + V * j) = q;
      } else if (j < a.half) {
        const int ia = a.pairs ? 2 * j : j, ib = a.pairs ? 2 * j + 1 : j + a.half;
        const float u = bf2f(src[ia]), v = bf2f(src[ib]);
        dst[ia] = f2bf(u * cs[0] - v * sn[0]);
        dst[ib] = f2bf(v * cs[0] + u * sn[0]);
      } else {
        dst[j + a.half] = src[j + a.half];
      }
    }
  }
}

// KC: steps of 32 inputs (K = 32 KC); CB: columns of the workgroup.  Of the grid's second dimension, the first H are the heads' products, the others
// the tails of TAIL_HEADS heads each, in small steps (one tile per workgroup) of 16 tokens each: sines are long chains of few threads there.
constexpr int TAIL_HEADS = 4;

template <int KC, int CB, bool GATE>
__global__ __launch_bounds__(NT, KC <= 4 ? 4 : 2) void heads_kernel(HeadArgs a) {
  constexpr int K = 32 * KC, LDW = K + 8;
  __shared__ __attribute__((aligned(16))) bf16_t Ws[CB * LDW];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), col = lane & 15, grp = lane >> 4;
  const int h = blockIdx.y, n0 = blockIdx.z * CB, t_first = blockIdx.x * a.tiles * 64, t_end = min(a.T, t_first + a.tiles * 64);
  if (h >= a.H) {
    if (blockIdx.z != 0) return;
    if (a.tiles == 1) {
      const int h0 = ((h - a.H) >> 2) * TAIL_HEADS, t0 = t_first + 16 * ((h - a.H) & 3);
      turn_tails<2>(a, K, t0, min(t_end, t0 + 16), h0, min(a.H, h0 + TAIL_HEADS));
    } else {
      const int h0 = (h - a.H) * TAIL_HEADS;
      turn_tails<8>(a, K, t_first, t_end, h0, min(a.H, h0 + TAIL_HEADS));
    }
    return;
  }
  const bf16_t* x = a.x + h * a.x_head;
  bf16x8 xf[KC];
  auto load = [&](int t0) {   // (rows past the end repeat the last one and are not stored)
    const bf16_t* p = x + static_cast<int64_t>(min(t0 + 16 * wave + col, a.T - 1)) * a.x_row + 8 * grp;
#pragma unroll
    for (int c = 0; c < KC; ++c) xf[c] = *reinterpret_cast<const bf16x8*>(p + 32 * c);
  };
  load(t_first);
  const bf16_t* w = a.w + static_cast<size_t>(h) * K * a.N + n0;
  for (int e = tid; e < (K / 4) * (CB / 4); e += NT) {   // 4 x 4 blocks; columns past N are not stored (N is a multiple of 16)
    const int n = 4 * (e % (CB / 4)), k = 4 * (e / (CB / 4));
    if (n0 + n >= a.N) continue;
    u16x4 r[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = *reinterpret_cast<const u16x4*>(w + static_cast<size_t>(k + i) * a.N + n);
#pragma unroll
    for (int j = 0; j < 4; ++j) *reinterpret_cast<u16x4*>(&Ws[(n + j) * LDW + k]) = u16x4{r[0][j], r[1][j], r[2][j], r[3][j]};
  }
  __syncthreads();
  for (int t0 = t_first; t0 < t_end; t0 += 64) {
    bf16x8 xc[KC];
#pragma unroll
    for (int c = 0; c < KC; ++c) xc[c] = xf[c];
    load(t0 + 64 < t_end ? t0 + 64 : t0);
    const int t = t0 + 16 * wave + col;
    s16x8 gq[GATE ? CB / 32 : 1];   // (asked for in front of the products)
    if constexpr (GATE) {
      const bf16_t* gp = a.gate + min(t, a.T - 1) * a.gate_row;
#pragma unroll
      for (int p = 0; p < CB / 32; ++p) {
        const int c = h * a.N + min(n0 + 16 * (2 * p + (grp & 1)) + 8 * (grp >> 1), a.N - 8);
        if (a.group == 1) gq[p] = *reinterpret_cast<const s16x8*>(gp + c);
        else gq[p][0] = static_cast<short>(gp[c / a.group]);   // (a multiple of 8: one column for all)
      }
    }
    // (the address passes through an empty statement: hipcc would keep all weights in 128 registers across the loop, two waves per SIMD)
    int w_at = col * LDW + 8 * grp;
    asm volatile("" : "+v"(w_at));
    f32x4 acc[CB / 16];
#pragma unroll
    for (int b = 0; b < CB / 16; ++b) {
      acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < KC; ++c) {
        const bf16x8 wf = *reinterpret_cast<const bf16x8*>(&Ws[w_at + 16 * b * LDW + 32 * c]);
        acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, xc[c], acc[b], 0, 0, 0);
      }
    }
#pragma unroll
    for (int p = 0; p < CB / 32; ++p) {
      // (lane groups 0 / 2 and 1 / 3 trade halves: eight neighbouring columns of block 2 p + (grp & 1) from 8 (grp >> 1) on)
      float o[8];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[2 * p][i]), __float_as_uint(acc[2 * p + 1][i]), false, false);
        o[i] = __uint_as_float(r[0]);
        o[4 + i] = __uint_as_float(r[1]);
      }
      const int n = n0 + 16 * (2 * p + (grp & 1)) + 8 * (grp >> 1);
      if (t >= t_end || n >= a.N) continue;
      s16x8 r;
      if constexpr (GATE) {
        float g[8];
        if (a.group == 1) {
#pragma unroll
          for (int i = 0; i < 8; ++i) g[i] = sigmoid(bf2f(static_cast<bf16_t>(gq[p][i])));
        } else {
          const float s = sigmoid(bf2f(static_cast<bf16_t>(gq[p][0])));
#pragma unroll
          for (int i = 0; i < 8; ++i) g[i] = s;
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) r[i] = static_cast<short>(f2bf(bf2f(f2bf(o[i])) * g[i]));
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) r[i] = static_cast<short>(f2bf(o[i]));
      }
      *reinterpret_cast<s16x8*>(a.out + static_cast<int64_t>(t) * a.o_row + h * a.o_head + n) = r;
    }
  }
}

template <int KC>
int launch(HeadArgs a, hipStream_t s) {
  // a workgroup turns its weight columns once: up to 512 tokens while four workgroups per CU are left
  const int64_t blocks = static_cast<int64_t>((a.T + 63) / 64) * a.H;
  a.tiles = static_cast<int>(std::min<int64_t>(8, std::max<int64_t>(1, blocks / 1024)));
  const int rows = (a.T + 64 * a.tiles - 1) / (64 * a.tiles);
  const bool wide = a.N > 64 && blocks >= 256;   // (few workgroups: 64 columns each, twice as many)
  const dim3 grid(rows, a.H + (a.n > 0 ? (a.H + TAIL_HEADS - 1) / TAIL_HEADS * (a.tiles == 1 ? 4 : 1) : 0), wide ? (a.N + 127) / 128 : (a.N + 63) / 64);
  if (a.gate != nullptr) {
    if (wide) heads_kernel<KC, 128, true><<<grid, NT, 0, s>>>(a);
    else heads_kernel<KC, 64, true><<<grid, NT, 0, s>>>(a);
  } else {
    if (wide) heads_kernel<KC, 128, false><<<grid, NT, 0, s>>>(a);
    else heads_kernel<KC, 64, false><<<grid, NT, 0, s>>>(a);
  }
  return BCG_CHECK_LAUNCH();
}

}  // namespace

// x [T, H, >= K] (strides in elements), w [H, K, N] contiguous, out [T, H, >= N]; K 32, 64, 128 or 256, N % 16 == 0; every pointer 16-byte aligned
// and every stride of x, out and (group 1) gate a multiple of 8.  n > 0: a tail of n features behind K and N; half: its turned pairs.
// gate (may be null): [T, H N / group] rows gate_row apart, group 1 or a multiple of 8 that divides N.
BCG_API int bcg_head_linear(const void* x, int64_t x_row, int64_t x_head, const void* w, void* out, int64_t o_row, int64_t o_head, int T_,
                            int H, int K, int N, const void* positions, const void* inv_freq, int n, int half, int pairs, float amp,
                            const void* gate, int64_t gate_row, int group, void* stream) {
  if (T_ <= 0) return 0;
  auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  if (H < 1 || H > 32767 || N < 16 || N % 16 || (N + 63) / 64 > 65535 || !al16(x) || !al16(w) || !al16(out) || x_row % 8 || x_head % 8 || o_row % 8 || o_head % 8) return -2;
  if (n < 0 || half < 0 || 2 * half > n || (n > 0 && (positions == nullptr || inv_freq == nullptr || gate != nullptr))) return -2;
  if (gate != nullptr && (group < 1 || (group == 1 ? gate_row % 8 != 0 || !al16(gate) : group % 8 != 0 || N % group != 0))) return -2;
  HeadArgs a;
  a.x = static_cast<const bf16_t*>(x); a.x_row = x_row; a.x_head = x_head;
  a.w = static_cast<const bf16_t*>(w);
  a.out = static_cast<bf16_t*>(out); a.o_row = o_row; a.o_head = o_head;
  a.T = T_; a.H = H; a.N = N; a.tiles = 1;
  a.positions = static_cast<const int*>(positions); a.inv_freq = static_cast<const float*>(inv_freq);
  a.n = n; a.half = half; a.pairs = pairs; a.amp = amp;
  a.gate = static_cast<const bf16_t*>(gate); a.gate_row = gate_row; a.group = group;
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (K) {
    case 32: return launch<1>(a, s);
    case 64: return launch<2>(a, s);
    case 128: return launch<4>(a, s);
    case 256: return launch<8>(a, s);
    default: return -2;
  }
}
