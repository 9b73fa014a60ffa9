// GEMM for tens to hundreds of rows (decode batches, short prefills): one workgroup per CU, the tile chosen so that one round of
// workgroups covers the product.
//
//   C[M, N] = X[M, K] · W[N, K]^T            (bf16 in, fp32 accumulate, bf16 out; F8: e4m3 in, scaled by row and column)
//
// What bounds it: W comes once from HBM, X out of L2 to every CU that holds a piece of W, and both go through a CU's one LDS-DMA path, which
// takes 114 B/ns where an instruction reads 128 bytes of a row and 77 where it reads 64 (1 KB each, L2 hits; 256 bytes: 112).  So:
//   * the waves split K, not the tile (WK = 4: a stage is 128 deep, wave w takes its w-th 32): every fragment is read out of LDS once,
//     (BM + BN) x 64 bytes a 32-deep step instead of the 1.5 times of 2 x 2 waves, which bound the 128 x 128 tiles of gemm.hip at 0.43 us per 64
//     of K.  Tiles of more than 40 blocks of 16 x 16 would need too many registers (four accumulators a block and lane): there, and where the
//     tile is wide from 32 on, WM = 2 halves of the rows, K in two;
//   * all four waves fetch an even share of X and W.  Two waves for X and two for W, with a deeper ring for W, took 1.3 times as long: a wave
//     has only so many fetches under way;
//   * the tile is free in steps of 16 (MID_TILES below: 3 to 16 blocks of rows by 1 to 12 of columns), so a plan (gemm_mid.hip) finds one whose
//     tiles x K-splits fill one round;
//   * the eight XCDs start K an eighth apart: in step, all CUs read the same 256 bytes of every row, a few channels' worth (101 x 24576 x 4096
//     48 -> 41 us); within an XCD they stay in step, so X and a W shared by several row tiles are fetched into its L2 once (a column tile whose row
//     tiles lie on two XCDs keeps the first one's start: equal rows stay equal);
//   * what runs once is kept short: a launch finds the instruction cache cold, and an unrolled epilogue of 10 KB took 4.2 us of fetches, this 2.2.
// Measured in a captured graph, other weights each call, us, tile kernels or library before -> here: 101 rows 24576 x 4096 gated 55 -> 45, 6144 x 4096
// 22.3 -> 20.4, 4096 x 4096 21 -> 15, 4096 x 12288 37 -> 35; 448 rows 5120 x 5120 51 -> 39, 5120 x 17408 109 -> 99, 6144 x 4096 47 -> 33;
// 96 rows 9728 x 896 gated 15 -> 10.  What is left at 101 rows: the first fetches take 2 us, the epilogue 1 to 2, a split's sum 3.
//
// LDS: rows of 128 bytes, the 16-byte chunk c of row r at c ^ ((r >> 1) & 7) (gemm.hip): fragment reads without conflicts, the swizzle applied to
// each lane's source.  Ring of R stages, one barrier per stage: a wave waits for its own fetches of stage s + 1, the barrier makes that
// everybody's (and everybody past the reads of stage s), then stage s + R goes into the slot of s and s + 1 into registers while the matrix
// products of s run.
#pragma once

#include <type_traits>

#include "common.h"

namespace {

// EPI_TAIL_GELU: gelu on the columns from `at` on, which go to an output of their own; EPI_GELU_TABLE: gelu times a row's entry of a table
enum Epilogue { EPI_STORE = 0, EPI_SILU_MUL = 1, EPI_RESIDUAL = 2, EPI_TAIL_GELU = 3, EPI_GELU_TABLE = 4 };
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef long i64x2 __attribute__((ext_vector_type(2)));

constexpr int LDS_BYTES = 163840;

struct MidArgs {
  const unsigned char *x, *w;
  const bf16_t *bias, *residual;
  bf16_t* c;
  float* ws;
  int* counters;
  const float *x_scale, *w_scale;
  int M, N, inter, blocks, m_tiles, n_tiles, split;   // inter: W's up rows behind its gate rows; blocks: of 128 bytes in a row of x and w
  bf16_t* tail;          // EPI_TAIL_GELU: [M, N - at]
  const bf16_t* table;   // EPI_GELU_TABLE: N columns of row tokens[m] (within 0 .. vocab - 1), rows `table_ld` apart
  const int* tokens;
  int at, table_ld, vocab;
};

__device__ __forceinline__ float silu(float g) { return g * __builtin_amdgcn_rcpf(1.f + __expf(-g)); }

// tanh form: z sigmoid(2 u) is 0.5 z (1 + tanh(u))
__device__ __forceinline__ float gelu(float z) {
  return z * __builtin_amdgcn_rcpf(1.f + __expf(-1.5957691216057308f * (z + 0.044715f * z * z * z)));
}

// buffer descriptor words (base, stride 0, num_records, raw-buffer config), wave-uniform
__device__ __forceinline__ i32x4 make_srd(const void* base, uint32_t bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(base);
  i32x4 r;
  r[0] = __builtin_amdgcn_readfirstlane(static_cast<int>(a & 0xffffffffu));
  r[1] = __builtin_amdgcn_readfirstlane(static_cast<int>(a >> 32) & 0xffff);
  r[2] = __builtin_amdgcn_readfirstlane(static_cast<int>(bytes));
  r[3] = 0x00020000;
  return r;
}

template <int N>
__device__ __forceinline__ void vm_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// MT x NT blocks of 16 x 16; WM: parts of the rows (each wave holds MT / WM of the row blocks and all column blocks)
template <int MT, int NT, int WM, int EPI, bool F8, bool SPLIT>
__global__ __launch_bounds__(256, 1) __attribute__((amdgpu_waves_per_eu(1, 1))) void gemm_mid_kernel(const MidArgs a) {
  constexpr int WK = 4 / WM;
  static_assert(WM == 1 || (WM == 2 && MT % 2 == 0 && NT % 2 == 0), "waves and fetches");
  static_assert(!F8 || EPI == EPI_STORE || EPI == EPI_RESIDUAL, "fp8: store / residual epilogues");
  static_assert(EPI != EPI_SILU_MUL || NT % 2 == 0, "gate and up blocks alternate");
  constexpr int U = MT + NT, MW = MT / WM, NB = MW * NT, F = MW + NT;
  static_assert(NB <= 64, "accumulators: the accumulation registers");
  constexpr int D = U * WK / 4;                 // fetches (1 KB) of a wave and stage
  constexpr int DX = D * MT / U;                // of these X's
  constexpr int STAGE = U * WK * 1024;
  constexpr int R = LDS_BYTES / STAGE > 6 ? 6 : LDS_BYTES / STAGE;
  static_assert(R >= 3 && (R - 2) * D <= 63, "ring");
  // ONE shared array: with a second one hipcc may wait for all fetches before every LDS read
  __shared__ __attribute__((aligned(1024))) unsigned char smem[LDS_BYTES];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kw = wave % WK, wm = wave / WK;

  // workgroups of one XCD: one K-split, neighbouring column tiles, their row tiles side by side
  const int nwg = a.m_tiles * a.n_tiles * a.split;
  const int bid = blockIdx.x, xcd = bid & 7, q = nwg >> 3, rem = nwg & 7;
  const int r_id = (xcd < rem ? xcd * (q + 1) : rem * (q + 1) + (xcd - rem) * q) + (bid >> 3);
  const int m_tile = r_id % a.m_tiles, rest = r_id / a.m_tiles;
  const int n_tile = rest % a.n_tiles, split = rest / a.n_tiles;
  const int width = EPI == EPI_SILU_MUL ? a.N / 2 : a.N, ld = EPI == EPI_SILU_MUL ? a.inter : EPI == EPI_TAIL_GELU ? a.at : a.N;   // columns written, of a row
  const int m0 = m_tile * MT * 16, n0 = n_tile * NT * (EPI == EPI_SILU_MUL ? 8 : 16);   // gated: the first feature
  const uint32_t row_bytes = static_cast<uint32_t>(a.blocks) * 128;
  const int kb0 = split * a.blocks / a.split, nb = (split + 1) * a.blocks / a.split - kb0;
  constexpr int H = WK / 2;                     // blocks of 128 bytes in a stage
  const int n = ((nb + H - 1) / H + 1) & ~1;    // stages, in pairs (registers of one step and the next)

  // rows past M / N and stages past the end fall outside the descriptors' range and read zeros
  i32x4 sX = make_srd(a.x + static_cast<size_t>(m0) * row_bytes, static_cast<uint32_t>(min(a.M - m0, MT * 16)) * row_bytes);
  i32x4 sW = make_srd(a.w + static_cast<size_t>(n0) * row_bytes,
                      EPI == EPI_SILU_MUL ? static_cast<uint32_t>(a.inter + min(width - n0, NT * 8)) * row_bytes
                                          : static_cast<uint32_t>(min(a.N - n0, NT * 16)) * row_bytes);
  const int range_x = sX[2], range_w = sW[2];
  // fetch u of a wave: 8 rows (group rg0 + u RG of X's, then W's) of one 128-byte block
  const int half = WK == 4 ? wave & 1 : 0;
  const int rg0 = WK == 4 ? wave >> 1 : wave;
  constexpr int RG = WK == 4 ? 2 : 4;
  const uint32_t v0 = (lane >> 3) * row_bytes + (((lane & 7) ^ (((rg0 & 1) * 4 + (lane >> 4)) & 7)) << 4);
  uint32_t vo[D];
#pragma unroll
  for (int u = 0; u < D; ++u) {
    const int r = (rg0 + u * RG - (u < DX ? 0 : 2 * MT)) * 8;
    // gated: 16 gate rows and 16 up rows of the same features alternate
    vo[u] = v0 + (EPI == EPI_SILU_MUL && u >= DX ? ((r >> 4) & 1) * a.inter + (r >> 5) * 16 + (r & 8) : r) * row_bytes;
  }
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem)) + half * U * 2048 + rg0 * 1024;
  // stage s of the walk is stage (s + rot) mod n of K.  rot: of the XCD that has the column tile's first row tile, so that rows of one call add K in
  // one order whichever row tile they are in (a column tile's row tiles may lie on two and more)
  int home = xcd;
  for (int from = r_id - (bid >> 3); r_id - m_tile < from; from -= home < rem ? q + 1 : q) --home;   // from: the first workgroup of `home`
  const int rot = home * n / 8;
  auto at = [&](int s) { const int t = s + rot; return t >= n ? t - n : t; };
  auto valid = [&](int s) { return s < n && at(s) * H + half < nb; };
  auto k_offset = [&](int s) { return __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(kb0 + at(s) * H + half) * 128); };
  // (s_nop: an LDS load needs a wait state behind a scalar write of m0, which hipcc does not put between instructions of one asm statement)
  auto fetch = [&](int u, uint32_t slot, uint32_t ko) {
    if (u < DX)
      asm volatile("s_add_u32 m0, %3, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(vo[u]), "s"(sX), "s"(ko), "s"(slot), "n"(u * RG * 1024) : "memory", "m0", "scc");
    else
      asm volatile("s_add_u32 m0, %3, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(vo[u]), "s"(sW), "s"(ko), "s"(slot), "n"(u * RG * 1024) : "memory", "m0", "scc");
  };
  auto aim = [&](int s) { sX[2] = valid(s) ? range_x : 0, sW[2] = valid(s) ? range_w : 0; };
  auto fetch_stage = [&](int s) {
    aim(s);
    const uint32_t ko = k_offset(s), slot = __builtin_amdgcn_readfirstlane(lds_base + s * STAGE);
#pragma unroll
    for (int u = 0; u < D; ++u) fetch(u, slot, ko);
  };

  const int fr = lane & 15, fq = lane >> 4;
  const unsigned char* rd = smem + (WK == 4 ? (kw >> 1) * U * 2048 : 0) + fr * 128 + ((((kw & 1) * 4 + fq) ^ (fr >> 1)) << 4);
  auto read = [&](const unsigned char* from, int f) {   // fragment f: X's row blocks of this wave, then W's
    return *reinterpret_cast<const bf16x8*>(from + (f < MW ? wm * MW + f : MT + f - MW) * 2048);
  };

  f32x4 acc[NT][MW];   // [column block][row block]: D[n = 4 fq + e][m = fr]
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MW; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 fa[F], fb[F];
  // (asm: with the builtin hipcc turns the accumulators over in copies.  Their first reader is behind the wait states after the loop.)
  auto product = [&](int p, const bf16x8 (&f)[F]) {
    const int i = p / MW, j = p % MW;
    if constexpr (F8) {   // the low and the high 8 bytes of every lane's 16: the same k in both operands
      const i64x2 w = __builtin_bit_cast(i64x2, f[MW + i]), x = __builtin_bit_cast(i64x2, f[j]);
      asm volatile("v_mfma_f32_16x16x32_fp8_fp8 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(w[0]), "v"(x[0]) : "memory");
      asm volatile("v_mfma_f32_16x16x32_fp8_fp8 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(w[1]), "v"(x[1]) : "memory");
    } else {
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(f[MW + i]), "v"(f[j]) : "memory");
    }
  };
  // product p and fetch u behind it, in one statement: the (first) product is the wait state between the write of m0 and the load.  Over 76
  // products 1.002 of the time with the write directly in front of the load, an s_nop between them 1.011 (up to 1.06 where a launch is short).
  auto product_fetch = [&](int p, const bf16x8 (&f)[F], int u, uint32_t slot, uint32_t ko) {
    const int i = p / MW, j = p % MW;
    const i32x4 srd = u < DX ? sX : sW;
    if constexpr (F8) {
      const i64x2 w = __builtin_bit_cast(i64x2, f[MW + i]), x = __builtin_bit_cast(i64x2, f[j]);
      const long w0 = w[0], w1 = w[1], x0 = x[0], x1 = x[1];
      asm volatile("s_add_u32 m0, %8, %9\n\tv_mfma_f32_16x16x32_fp8_fp8 %0, %1, %2, %0\n\tbuffer_load_dwordx4 %5, %6, %7 offen lds\n\t"
                   "v_mfma_f32_16x16x32_fp8_fp8 %0, %3, %4, %0"
                   : "+a"(acc[i][j])
                   : "v"(w0), "v"(x0), "v"(w1), "v"(x1), "v"(vo[u]), "s"(srd), "s"(ko), "s"(slot), "n"(u * RG * 1024)
                   : "memory", "m0", "scc");
    } else {
      asm volatile("s_add_u32 m0, %6, %7\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %2, %0\n\tbuffer_load_dwordx4 %3, %4, %5 offen lds"
                   : "+a"(acc[i][j])
                   : "v"(f[MW + i]), "v"(f[j]), "v"(vo[u]), "s"(srd), "s"(ko), "s"(slot), "n"(u * RG * 1024)
                   : "memory", "m0", "scc");
    }
  };

#pragma unroll
  for (int s = 0; s < R - 1; ++s) fetch_stage(s);
  vm_wait<(R - 2) * D>();
  __builtin_amdgcn_s_barrier();
  fetch_stage(R - 1);
#pragma unroll
  for (int f = 0; f < F; ++f) fa[f] = read(rd, f);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  uint32_t rslot = STAGE, wslot = 0;            // slots of stages s + 1 and s + R
  constexpr int EV = F > D ? F : D;             // memory operations of a step, spread over the first PE of its products
  constexpr int PE = NB < EV ? NB : NB - NB / 8;
  auto step = [&](int s, bf16x8 (&cur)[F], bf16x8 (&nxt)[F]) {
    vm_wait<(R - 2) * D>();
    __builtin_amdgcn_s_barrier();
    aim(s + R);
    const uint32_t ko = k_offset(s + R), slot = __builtin_amdgcn_readfirstlane(lds_base + wslot);
    const unsigned char* from = rd + rslot;
    __builtin_amdgcn_sched_barrier(0);
    auto walk = [&](auto self, auto pp) {
      constexpr int p = decltype(pp)::value;
      if constexpr (p < NB) {
        constexpr int next = ((p + 1) * EV + PE - 1) / PE, last = (next < EV ? next : EV) - 1;   // the last operation in front of this product
        auto ops = [&](auto self2, auto ee) {
          constexpr int e = decltype(ee)::value;
          if constexpr (e < EV && e * PE / EV <= p) {
            if constexpr (e * PE / EV == p) {
              if constexpr (e < F) nxt[e] = read(from, e);
              if constexpr (e < D && e != last) fetch(e, slot, ko);
              __builtin_amdgcn_sched_barrier(0);
            }
            self2(self2, std::integral_constant<int, e + 1>{});
          }
        };
        ops(ops, std::integral_constant<int, (p * EV + PE - 1) / PE>{});
        if constexpr (last * PE / EV == p && last < D)
          product_fetch(p, cur, last, slot, ko);
        else
          product(p, cur);
        __builtin_amdgcn_sched_barrier(0);
        self(self, std::integral_constant<int, p + 1>{});
      }
    };
    walk(walk, std::integral_constant<int, 0>{});
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    rslot = rslot + STAGE == R * STAGE ? 0 : rslot + STAGE;
    wslot = wslot + STAGE == R * STAGE ? 0 : wslot + STAGE;
  };
  int s = 0;
  do {   // (a split holds a block at least: two stages)
    step(s, fa, fb);
    step(s + 1, fb, fa);
    s += 2;
  } while (s < n);
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_nop 15\n\ts_nop 15" ::: "memory");

  // ---- sum over the K-waves and epilogue, by rows: [kw][row][BN + 4] of LDS (BN / 4 + 1 is odd: the 16 rows of a store hit 16 slots),
  // then 8 columns a lane.  Row blocks in PH phases where the tile does not fit.
  constexpr int BN = NT * 16, LROW = BN + 4;
  constexpr int JC = LDS_BYTES / (256 * LROW) < MW ? LDS_BYTES / (256 * LROW) : MW;
  constexpr int PH = (MW + JC - 1) / JC, JP = (MW + PH - 1) / PH;
  constexpr int CI = EPI == EPI_SILU_MUL ? NT : NT * 2;   // items (8 columns of the output) of a row
  constexpr int IT = (WM * JP * 16 * CI + 255) / 256;     // items of a thread and phase
  constexpr int Q = EPI == EPI_SILU_MUL ? 4 : 2;          // groups of 4 sums of an item
  constexpr int SLAB = MT * 16 * BN;                      // floats of a split's part
  float* red = reinterpret_cast<float*>(smem);
  const int tile = n_tile * a.m_tiles + m_tile;
  const uint32_t ldb = static_cast<uint32_t>(ld) * 2;
  const size_t corner = static_cast<size_t>(m0) * ld;
  const int rows = min(a.M - m0, MT * 16);                // of the tile in the output
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(SPLIT ? a.ws + static_cast<size_t>(tile) * a.split * SLAB : a.ws, 0,
                                                                      SPLIT ? a.split * SLAB * 4 : 0, 0x00020000);
  const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(a.c + corner, 0, rows * ldb, 0x00020000);
  const __amdgpu_buffer_rsrc_t rr = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(EPI == EPI_RESIDUAL ? a.residual + corner : a.c), 0,
                                                                      EPI == EPI_RESIDUAL ? rows * ldb : 0, 0x00020000);
  const uint32_t ldt = static_cast<uint32_t>(EPI == EPI_TAIL_GELU ? a.N - a.at : 0) * 2;
  const __amdgpu_buffer_rsrc_t rt = __builtin_amdgcn_make_buffer_rsrc(EPI == EPI_TAIL_GELU ? a.tail + static_cast<size_t>(m0) * (a.N - a.at) : a.c, 0,
                                                                      rows * ldt, 0x00020000);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(a.bias), 0, a.bias ? ldb : 0, 0x00020000);
  struct Item {
    uint32_t off, boff;   // bytes from the tile's corner, from the row's start
    bf16x8 r, b;
    float xs;
    f32x4 ws[2];
    bool tail;
  };
  auto load8 = [&](const __amdgpu_buffer_rsrc_t& rsrc, uint32_t off) { return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, 0, 0)); };
  // (past the rows or the width an offset past every range: stores are dropped, loads are 0)
  auto place = [&](int row, int ci) {
    Item t;
    const int c = n0 + ci * 8;
    t.boff = c < width ? c * 2 : 0x80000000u;
    t.tail = EPI == EPI_TAIL_GELU && c >= a.at;   // (at is a multiple of 8: an item lies on one side)
    t.off = c < width && row < rows ? t.tail ? row * ldt + (c - a.at) * 2 : row * ldb + c * 2 : 0x80000000u;
    return t;
  };
  auto load = [&](Item& t, int row) {
    if constexpr (EPI == EPI_RESIDUAL) t.r = load8(rr, t.off);
    if constexpr (EPI == EPI_GELU_TABLE) {
      const int token = min(max(a.tokens[m0 + min(row, rows - 1)], 0), a.vocab - 1);
      t.r = *reinterpret_cast<const bf16x8*>(a.table + static_cast<size_t>(token) * a.table_ld + min(t.boff >> 1, static_cast<uint32_t>(width) - 8));
    }
    if constexpr (EPI == EPI_STORE || EPI == EPI_RESIDUAL) t.b = load8(rb, t.boff);
    if constexpr (F8) {
      t.xs = a.x_scale[m0 + min(row, rows - 1)];
      const f32x4* p = reinterpret_cast<const f32x4*>(a.w_scale + min(t.boff >> 1, static_cast<uint32_t>(width) - 8));
      t.ws[0] = p[0], t.ws[1] = p[1];
    }
  };
  auto finish = [&](const Item& t, const f32x4 (&v)[Q]) {
    bf16x8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float y = v[e >> 2][e & 3];
      if constexpr (EPI == EPI_SILU_MUL) {
        y = silu(y) * v[2 + (e >> 2)][e & 3];
      } else if constexpr (EPI == EPI_GELU_TABLE) {
        y = gelu(y) * static_cast<float>(t.r[e]);
      } else if constexpr (EPI == EPI_TAIL_GELU) {
        if (t.tail) y = gelu(y);
      } else {
        if constexpr (F8) y *= t.xs * t.ws[e >> 2][e & 3];
        y += static_cast<float>(t.b[e]);
        if constexpr (EPI == EPI_RESIDUAL) y += static_cast<float>(t.r[e]);
      }
      o[e] = static_cast<__bf16>(y);
    }
    if (EPI == EPI_TAIL_GELU && t.tail) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, o), rt, t.off, 0, 0);
    else __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, o), rc, t.off, 0, 0);
  };
#pragma unroll
  for (int ph = 0; ph < PH; ++ph) {
    const int j0 = ph * JP, jn = MW - j0 < JP ? MW - j0 : JP;
    const int held = WM * jn * 16;                        // rows of this phase: jn row blocks of every part
    auto row_of = [&](int lr) { const int g = lr / (jn * 16); return (g * MW + j0) * 16 + lr - g * jn * 16; };
    Item it[IT];
#pragma unroll
    for (int t = 0; t < IT; ++t) {
      const int id = tid + t * 256, lr = id / CI, row = row_of(lr);
      it[t] = place(lr < held ? row : rows, id % CI);
      if constexpr (!SPLIT) load(it[t], row);
    }
    __syncthreads();
#pragma unroll
    for (int j = j0; j < j0 + jn; ++j)
#pragma unroll
      for (int i = 0; i < NT; ++i)
        *reinterpret_cast<f32x4*>(red + ((kw * WM + wm) * jn * 16 + (j - j0) * 16 + fr) * LROW + i * 16 + fq * 4) = acc[i][j];
    __syncthreads();
#pragma unroll
    for (int t = 0; t < IT; ++t) {
      const int id = tid + t * 256, lr = min(id / CI, held - 1), ci = id % CI;
      f32x4 v[Q];
#pragma unroll
      for (int g = 0; g < Q; ++g) {
        const float* from = red + lr * LROW + (EPI == EPI_SILU_MUL ? (ci >> 1) * 32 + (ci & 1) * 8 + (g >> 1) * 16 + (g & 1) * 4 : ci * 8 + g * 4);
        v[g] = *reinterpret_cast<const f32x4*>(from);
#pragma unroll
        for (int w = 1; w < WK; ++w) v[g] += *reinterpret_cast<const f32x4*>(from + w * held * LROW);
      }
      if constexpr (!SPLIT) {
        finish(it[t], v);
      } else {
        const int row = row_of(lr);
        const uint32_t so = id / CI < held && row < rows ? (split * SLAB + (row * CI + ci) * (Q * 4)) * 4 : 0x80000000u;
#pragma unroll
        for (int g = 0; g < Q; ++g) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v[g]), rs, so + g * 16, 0, 16 /*sc1*/);
      }
    }
  }
  if constexpr (!SPLIT) return;

  // ---- K split over workgroups: the last one to arrive adds the parts (write-through stores, one ticket: gemm.hip), always in the order of
  // the splits.  All loads of a batch first: with four splits one after another this took 6 us, so 3.
  vm_wait<0>();
  __syncthreads();
  int* flag = reinterpret_cast<int*>(smem);
  if (tid == 0) {
    const int prev = __hip_atomic_fetch_add(&a.counters[tile], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int last = prev == a.split - 1;
    if (last) __hip_atomic_store(&a.counters[tile], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // next launch
    flag[0] = last;
  }
  __syncthreads();
  if (!flag[0]) return;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");  // no instruction: keeps the loads below
  constexpr int B = 8 / Q;                                // items of a thread in flight
  const int items = rows * CI;
#pragma unroll 1
  for (int t0 = tid; t0 < items; t0 += 256 * B) {
    f32x4 v[B][Q];
    Item it[B];
#pragma unroll
    for (int b = 0; b < B; ++b) {
      const int id = t0 + b * 256;
      it[b] = place(id / CI, id % CI);
      load(it[b], id / CI);
#pragma unroll
      for (int g = 0; g < Q; ++g) v[b][g] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll 1
    for (int s0 = 0; s0 < a.split; s0 += 4) {             // (parts past the last are past the range: zeros)
      u32x4 l[4][B][Q];
#pragma unroll
      for (int sp = 0; sp < 4; ++sp)
#pragma unroll
        for (int b = 0; b < B; ++b)
#pragma unroll
          for (int g = 0; g < Q; ++g) {
            const int id = t0 + b * 256;
            l[sp][b][g] = __builtin_amdgcn_raw_buffer_load_b128(rs, id < items ? ((s0 + sp) * SLAB + id * (Q * 4) + g * 4) * 4 : 0x80000000u, 0, 16);
          }
#pragma unroll
      for (int sp = 0; sp < 4; ++sp)
#pragma unroll
        for (int b = 0; b < B; ++b)
#pragma unroll
          for (int g = 0; g < Q; ++g) v[b][g] += __builtin_bit_cast(f32x4, l[sp][b][g]);
    }
#pragma unroll
    for (int b = 0; b < B; ++b) finish(it[b], v[b]);
  }
}

// Of 72 tiles that were timed, those without which the choice by `predicted` would be slower (28: 0.3 % behind all of them on average).
#define MID_TILES(T) \
  T(0, 3, 1, 1) T(1, 3, 2, 1) T(2, 3, 3, 1) T(3, 3, 4, 1) T(4, 3, 6, 1) T(5, 4, 2, 1) \
  T(6, 4, 3, 1) T(7, 4, 4, 1) T(8, 4, 5, 1) T(9, 5, 4, 1) T(10, 5, 5, 1) T(11, 5, 6, 1) \
  T(12, 6, 4, 1) T(13, 6, 6, 1) T(14, 8, 4, 1) T(15, 8, 5, 1) T(16, 4, 8, 2) T(17, 4, 10, 2) \
  T(18, 6, 8, 2) T(19, 6, 10, 2) T(20, 8, 6, 2) T(21, 8, 10, 2) T(22, 10, 6, 2) T(23, 10, 8, 2) \
  T(24, 10, 12, 2) T(25, 12, 10, 2) T(26, 14, 8, 2) T(27, 16, 8, 2)

template <int EPI, bool F8>
int launch(int tile, const MidArgs& a, hipStream_t stream) {
  const dim3 grid(a.m_tiles * a.n_tiles * a.split);
  switch (tile) {
#define T(i, m, n, w)                                                                                           \
  case i:                                                                                                       \
    if constexpr (EPI != EPI_SILU_MUL || (n) % 2 == 0) {                                                        \
      if (a.split > 1)                                                                                          \
        hipLaunchKernelGGL((gemm_mid_kernel<m, n, w, EPI, F8, true>), grid, dim3(256), 0, stream, a);           \
      else                                                                                                      \
        hipLaunchKernelGGL((gemm_mid_kernel<m, n, w, EPI, F8, false>), grid, dim3(256), 0, stream, a);          \
      return BCG_CHECK_LAUNCH();                                                                                \
    }                                                                                                           \
    return -2;
    MID_TILES(T)
#undef T
  }
  return -2;
}

}  // namespace
