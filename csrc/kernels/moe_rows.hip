// Expert products of a small step: per position tile of at most 32 rows (one expert) C = A W_e^T, bf16.
//
// What bounds it: a decode step gives an expert a handful of rows (64 tokens x 2 of 8 experts: 16), so its weight is streamed
// once for few rows and the kernel is the few-row projection (gemm_skinny.hip, which says why its loads and shares are as they are) with two
// differences: a workgroup belongs to a position tile, S workgroups share the rows of its expert's weight, and rows of A are
// gathered by the slots of the tile.  8 experts of 4096 (gated pairs) x 2048 and 2048 x 2048, 128 slots: 53 and 40 us with the 64 x 64 tile
// kernel (2.5 and 1.7 TB/s: 640 and 320 workgroups of short K-loops behind barriers), 30 and 16 here; align, both products and combine
// 97 -> 54.
#include <type_traits>

#include "seqmix_common.h"

namespace {

constexpr int NW = 8, MT = 2, NT = 4, TILE = 16 * MT;   // waves, blocks of 16 rows of A and of W
constexpr uint32_t PAST_END = 0x80000000u;              // an offset outside every descriptor
constexpr int RELU2 = 1, GATED = 2;                     // `ACT` classes: 0 none, 1 squared relu, 2 gated pairs (act 2 and 3)

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct MoeRowsArgs {
  const uint8_t* a;        // [rows, K]
  const uint8_t* w;        // [E, N, K]
  bf16_t* out;
  const int* sorted;       // [tiles * TILE] slot of a position, -1: none
  const int* tile_expert;  // [tiles], -1: unused
  int64_t out_stride;
  uint32_t a_bytes, a_step;   // bytes of a, of one of its rows
  int row_bytes, N, top, gather, scatter, act, shares;
  float limit;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}

// ACT == GATED: W's rows alternate 16 gate and 16 up rows of the same features.
template <int ACT>
__global__ __launch_bounds__(64 * NW, 2) void moe_rows_kernel(MoeRowsArgs p) {
  constexpr int PAIR = ACT == GATED ? 2 : 1, OUT = NT / PAIR * MT, PART = OUT * PAIR * 1024;
  __shared__ __attribute__((aligned(16))) uint8_t smem[NW * PART];
  const int tile = blockIdx.x / p.shares, share = blockIdx.x % p.shares;
  const int expert = p.tile_expert[tile];
  if (expert < 0) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, kg = lane >> 4;
  const uint32_t rb = p.row_bytes;
  // this workgroup's blocks of 16 output columns, in passes of NT / PAIR
  const int blocks = p.N / (16 * PAIR), b0 = blocks * share / p.shares, nb = blocks * (share + 1) / p.shares - b0;
  const int passes = (nb + NT / PAIR - 1) / (NT / PAIR);
  if (passes == 0) return;
  const int per = (nb + passes - 1) / passes;
  const int nu = (rb + 255) / 256, lw = (nu + NW - 1) / NW;   // units of K, a wave's units of a pass
  const uint32_t half = (rb & 255) && kg >= 2 ? PAST_END : 0;  // the last unit may be half a unit
  const uint32_t chunk = kg * 64 + (lane & 3) * 16;
  const uint32_t vo = ((lane >> 2) & 3) * 4 * rb + chunk;
  const uint8_t* wb = p.w + (static_cast<size_t>(expert) * p.N + static_cast<size_t>(b0) * 16 * PAIR) * rb;
  const __amdgpu_buffer_rsrc_t ar = rsrc(p.a, p.a_bytes);
  uint32_t xo[MT][4];   // rows of A that load i of a block takes in this lane
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int pos = tile * TILE + m * 16 + ((lane >> 2) & 3) * 4 + i, slot = p.sorted[pos];
      xo[m][i] = slot < 0 ? PAST_END : static_cast<uint32_t>(p.gather ? slot / p.top : pos) * p.a_step + chunk;
    }

  u32x4 wf[NT][4], xf[MT][4];
  struct Item {
    int p, j;
  };
  struct Where {
    const uint8_t* w;
    int bytes;
    uint32_t off, past;   // past: of this lane, PAST_END where nothing is to be read
  };
  auto advance = [&](Item& it) {
    if (++it.j == lw) {
      it.j = 0;
      ++it.p;
    }
  };
  auto where = [&](Item it) {
    const int t = wave + it.j * NW;
    const bool in = t < nu && it.p < passes;
    const int off = in ? t * 256 : 0, first = in ? it.p * per : 0;
    return Where{wb + static_cast<size_t>(first) * 16 * PAIR * rb + off,
                 in ? min(per, nb - first) * 16 * PAIR * static_cast<int>(rb) - off : 0, static_cast<uint32_t>(off),
                 in ? (t + 1 == nu ? half : 0) : PAST_END};
  };
  auto load_x = [&](const Where& at, int m) {
#pragma unroll
    for (int i = 0; i < 4; ++i) xf[m][i] = __builtin_amdgcn_raw_buffer_load_b128(ar, (xo[m][i] + at.off) | at.past, 0, 0);
  };
  auto load_w = [&](const Where& at, int n) {
    const int skip = n * 16 * static_cast<int>(rb);
    const __amdgpu_buffer_rsrc_t rs = rsrc(at.w + skip, max(at.bytes - skip, 0));
#pragma unroll
    for (int i = 0; i < 4; ++i) wf[n][i] = __builtin_amdgcn_raw_buffer_load_b128(rs, (vo + i * rb) | at.past, 0, 2 /*nt*/);
  };
  f32x4 acc[NT][MT];
  auto clear = [&] {
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  auto finish = [&](int pass) {
#pragma unroll
    for (int o = 0; o < OUT; ++o)
#pragma unroll
      for (int h = 0; h < PAIR; ++h)
        *reinterpret_cast<f32x4*>(smem + wave * PART + (o * PAIR + h) * 1024 + lane * 16) = acc[o / MT * PAIR + h][o % MT];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    auto total = [&](int blk) {
      f32x4 v = *reinterpret_cast<const f32x4*>(smem + blk * 1024 + lane * 16);
#pragma unroll
      for (int w = 1; w < NW; ++w) v += *reinterpret_cast<const f32x4*>(smem + w * PART + blk * 1024 + lane * 16);
      return v;
    };
    for (int o = wave; o < OUT; o += NW) {
      const int i = o / MT, pos = tile * TILE + (o % MT) * 16 + r, blk = pass * per + i;
      const int slot = p.sorted[pos];
      if (i >= per || blk >= nb || slot < 0) continue;
      f32x4 v = total(o * PAIR);
      u16x4 q;
      if constexpr (ACT == GATED) {
        const f32x4 up = total(o * PAIR + 1);
#pragma unroll
        for (int e = 0; e < 4; ++e) q[e] = gated_hidden<bf16_t>(v[e], up[e], p.act, p.limit);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (ACT == RELU2) {
            v[e] = fmaxf(v[e], 0.f);
            v[e] *= v[e];
          }
          q[e] = f2bf(v[e]);
        }
      }
      *reinterpret_cast<u16x4*>(p.out + static_cast<int64_t>(p.scatter ? slot : pos) * p.out_stride + (b0 + blk) * 16 + 4 * kg) = q;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();   // before the next pass's partial tiles
  };

  Item now{0, 0}, next{0, 0};
  {
    const Where at = where(next);
    advance(next);
#pragma unroll
    for (int m = 0; m < MT; ++m) load_x(at, m);
#pragma unroll
    for (int n = 0; n < NT; ++n) load_w(at, n);
  }
  clear();
  while (true) {
    const Where at = where(next);
    advance(next);
    u32x4 xt[MT][4];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      quad_transpose(xf[m], xt[m]);
      load_x(at, m);
      __builtin_amdgcn_sched_barrier(0);   // a register is loaded again where it was consumed, not later
    }
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      u32x4 wt[4];
      quad_transpose(wf[n], wt);
      load_w(at, n);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int m = 0; m < MT; ++m)
          acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wt[j]), __builtin_bit_cast(bf16x8, xt[m][j]),
                                                               acc[n][m], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (now.j + 1 == lw) {
      finish(now.p);
      if (now.p + 1 == passes) return;
      clear();
    }
    advance(now);
  }
}

}  // namespace

BCG_API int bcg_moe_rows_tile() { return TILE; }

// One product of `tiles` position tiles of bcg_moe_rows_tile() rows (bcg_moe_align).  a: [a_rows, K] bf16, rows a_stride apart; row of a
// position: its slot / top (gather) or the position itself; output row: the slot (scatter) or the position.  act 0 none, 1 squared
// relu, 2 and 3 gated (N rows in pairs, N / 2 output columns).  K % 64 == 0, N % 16 == 0 (gated: 32); 16-byte aligned.
// tiles: no fewer than hold rows (they come first); experts: how many are likely to (the launch splits the weights for that many: all
// workgroups that have work at once on 256 CUs, one each).
BCG_API int bcg_moe_rows(const void* a, int64_t a_rows, int64_t a_stride, const void* w, void* out, int64_t out_stride, const void* sorted,
                         const void* tile_expert, int tiles, int experts, int N, int K, int top, int gather, int scatter, int act,
                         float limit, void* stream) {
  if (tiles <= 0) return 0;
  if (K < 64 || K % 64 || K > 32768 || act < 0 || act > 3 || N < 1 || N % (act >= 2 ? 32 : 16) || top < 1 || experts < 1 ||
      a_stride < K || a_stride % 8 || out_stride % 4 || a_rows * a_stride * 2 >= (1LL << 31))
    return -2;
  const int blocks = N / (act >= 2 ? 32 : 16);
  int shares = 256 / experts;
  shares = shares < 1 ? 1 : shares > blocks ? blocks : shares;
  if (static_cast<int64_t>(tiles) * shares > (1 << 24)) return -2;
  const MoeRowsArgs p{static_cast<const uint8_t*>(a), static_cast<const uint8_t*>(w), static_cast<bf16_t*>(out),
                      static_cast<const int*>(sorted), static_cast<const int*>(tile_expert), out_stride,
                      static_cast<uint32_t>(a_rows * a_stride * 2), static_cast<uint32_t>(a_stride * 2), 2 * K, N, top, gather, scatter, act,
                      shares, limit};
  const dim3 grid(tiles * shares), block(64 * NW);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (act >= 2)
    moe_rows_kernel<GATED><<<grid, block, 0, s>>>(p);
  else if (act == 1)
    moe_rows_kernel<RELU2><<<grid, block, 0, s>>>(p);
  else
    moe_rows_kernel<0><<<grid, block, 0, s>>>(p);
  return BCG_CHECK_LAUNCH();
}
