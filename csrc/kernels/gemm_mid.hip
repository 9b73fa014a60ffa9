// Plan and entry points of gemm_mid.h; each epilogue's kernels are a source of their own (they compile side by side).
#include "gemm_mid.h"

BCG_API int bcg_gemm_mid_gated(int tile, const void* args, hipStream_t stream);
BCG_API int bcg_gemm_mid_residual(int tile, const void* args, hipStream_t stream);
BCG_API int bcg_gemm_mid_fp8(int tile, const void* args, hipStream_t stream);
BCG_API int bcg_gemm_mid_fp8_residual(int tile, const void* args, hipStream_t stream);
BCG_API int bcg_gemm_mid_tail_gelu(int tile, const void* args, hipStream_t stream);
BCG_API int bcg_gemm_mid_gelu_table(int tile, const void* args, hipStream_t stream);

namespace {

struct MidTile {
  int mt, nt, wm;
};
constexpr MidTile TILES[] = {
#define T(i, m, n, w) {m, n, w},
    MID_TILES(T)
#undef T
};
constexpr int N_TILES = sizeof(TILES) / sizeof(TILES[0]);
constexpr int CUS = 256;

// Microseconds of a launch of one round, x_rows rows of X (a row tile's share) and bn of W, kb bytes each, a workgroup: fitted (relative least squares,
// three ranges of rows) to the times of these tiles at 2300 products and checked at 1600 others: the tile chosen by it is 1.7, 2.3 and
// 3.2 % slower on average than the best of all 72.  (The times are not kept: for another compiler or card, time bcg_gemm_mid with every tile and
// split of random products, weights changed each call, and fit the nine terms of `predicted` again.)
struct Cost {
  float launch, x_row, w_row, product, hbm, area, split, part, gated_part;
};
constexpr Cost COSTS[] = {{3.1f, 10.f, 11.9f, 75.5f, 29.2f, 1.73f, 2.3f, 7.8f, 15.5f},      // up to 128 rows
                          {3.0f, 8.5f, 11.6f, 55.5f, 37.1f, 1.77f, 2.65f, 8.5f, 17.3f},     // up to 288
                          {2.75f, 9.6f, 10.6f, 43.4f, 47.4f, 1.93f, 3.3f, 9.f, 17.8f}};
float predicted(const Cost& c, float x_rows, int bm, int bn, float kb, float w_bytes, int split, bool gated, bool f8) {
  const float area = static_cast<float>(bm) * bn;
  const float t = c.launch + (c.x_row * x_rows + c.w_row * bn) * kb * 1e-6f + c.product * area * kb * (f8 ? 1e-9f : 0.5e-9f) +
                  c.hbm * w_bytes * (1e-6f / CUS) + c.area * area * 1e-4f;
  return split == 1 ? t : t + c.split + (gated ? c.gated_part : c.part) * split * area * 1e-5f;
}

}  // namespace

// How x [M, K] w [N, K]^T runs here: tile | split << 8, or -1 where it does not: the product has to fit one round of workgroups
// (several rounds lose to the persistent 256 x 256 kernel).  W holds 0.1 M elements or more: 603 products of 0.1 to 0.8 M and K >= 192 took 0.67 of
// the library's or few-row kernel's time on average, the slowest 1.06, 1.10 and 1.14 (92 x 96 x 1536, 182 x 96 x 1152 and 57 x 256 x 2048, 4.7 to
// 5.5 us), all others up to 1.04; of 64 and 128 columns of K it is 0.8 M (below, up to 1.17 of a library launch of 4 to 5 us), of fp8 0.8 M.
// 33 to 1024 rows, 900 products of 64 to 40000 columns and K of 256 to 18000, this over what took
// them before (tile kernels, library, few-row kernel): up to 64 rows 0.65, 128: 0.66, 256: 0.70, 512: 0.73, 1024: 0.84 on average; 12 projections of the
// served models 0.81 to 0.90, the slowest (40 to 64 rows, 7168 x 5120 and 6144 x 4096) 1.1.  fp8, whose other side has matrix
// instructions of twice the rate: 0.5 to 0.86, but 0.8 to 1.25 from M N K = 15e9 on; bf16 1.0 to 1.18 from 80e9 on.
// 1025 to 1536 rows, 213 products of more than 512 columns: 0.86 on average, the slowest 1.03; then the library's tiles fill the chip as well: 0.87
// and 1.07 to 1792 rows, 0.93 and 1.05 to 2047, where 2048 x 8192 behind 2039 rows took 80 us for 70.  Up to 512 columns the library's split of a
// long K wins at times (1508 x 256 x 5632: 22.5 us for 18.3).  fp8 past 1024 rows 0.64 to 0.95 on average, but 1.2 to 1.33 at 768 to 1792
// columns of K, which nothing here tells apart.
// What else is left to the others (times over theirs): bf16, plain, K of 64 or, up to 128 rows, of 128 into a store (67 products of 6000 to 40000
// columns: 0.72 to 0.96 on average, but 11 of 1.05 to 1.25); plain, up to 128 rows and 144 columns, K below 2304 (37: 0.91, 12 of 1.03 to 1.16; past
// these lines 0.48 to 0.87 and 1 of 143).  fp8 into a store, where the other side is one library launch (into a residual it is two: 0.49 to 0.77): K of 128
// (38 products: 0.98, 18 of 1.03 to 1.19), K of 256 with 65 to 256 rows (29: 0.93, 13), and from M N K = 1.5e9 on more than 176 rows with K up to
// 3600 (0.97, 40 of 1.03 to 1.4, where its 128 x 128 tiles fill the chip, which nothing here tells); the 281 that stay 0.74 on average, 11 of 1.03 to 1.21.
BCG_API int bcg_gemm_mid_plan(int epi, int M, int N, int K, int f8) {
  const bool gated = epi == EPI_SILU_MUL;
  const int bytes = f8 ? K : 2 * K, inter = N / 2;
  if (M < 33 || M > (f8 ? 1024 : 1536) || (M > 1024 && N <= 512) || K <= 0 || bytes % 128 || N < 16 || N % (gated ? 32 : 16) || N > 1 << 20 || (f8 && gated)) return -1;
  if (static_cast<int64_t>(N) * K < (f8 || K < 192 ? 800000 : 100000) || static_cast<int64_t>(N) * bytes >= 1ll << 31 || static_cast<int64_t>(M) * bytes >= 1ll << 31) return -1;
  const Cost& cost = COSTS[M <= 128 ? 0 : M <= 288 ? 1 : 2];
  const float products = static_cast<float>(M) * N * K;
  if (products > (f8 ? 15e9f : 80e9f)) return -1;
  if (f8 && epi == EPI_STORE && (K == 128 || (K == 256 && M > 64 && M <= 256) || (M > 176 && K <= 3600 && products >= 1.5e9f))) return -1;
  if (!f8 && epi == EPI_STORE && (K == 64 || (K == 128 && M <= 128))) return -1;
  if (!f8 && !gated && M <= 128 && N <= 144 && K < 2304) return -1;
  int best = -1;
  float time = 0.f;
  for (int i = 0; i < N_TILES; ++i) {
    const int bm = TILES[i].mt * 16, bn = TILES[i].nt * 16;
    if (gated && TILES[i].nt % 2) continue;
    const int m_tiles = (M + bm - 1) / bm, tiles = m_tiles * (gated ? (inter + bn / 2 - 1) / (bn / 2) : (N + bn - 1) / bn);
    if (tiles > CUS) continue;
    for (int split : {1, 2, 3, 4, 6, 8}) {
      // (four of K's 128-byte blocks a split: fewer are all start and end)
      if (split > 1 && (tiles * split > CUS || bytes / 128 < 4 * split)) break;
      const float t = predicted(cost, static_cast<float>(M) / m_tiles, bm, bn, static_cast<float>(bytes) / split, static_cast<float>(N) * bytes, split, gated, f8);
      if (best < 0 || t < time) best = i | split << 8, time = t;
    }
  }
  return best;
}

// fp32 parts (floats of `ws`) and arrival counters (ints, 0 before and after every launch) of a plan; 0 and 0 without a split
BCG_API int64_t bcg_gemm_mid_parts(int plan, int epi, int M, int N, int* tiles) {
  const MidTile t = TILES[plan & 255];
  const int bn = t.nt * 16, width = epi == EPI_SILU_MUL ? N / 2 : N, cols = epi == EPI_SILU_MUL ? bn / 2 : bn;
  *tiles = (M + t.mt * 16 - 1) / (t.mt * 16) * ((width + cols - 1) / cols);
  return plan >> 8 > 1 ? static_cast<int64_t>(*tiles) * (plan >> 8) * t.mt * 16 * bn : 0;
}

// Number of the capture that records what is launched on the stream (no two have the same), 0 without one
BCG_API int64_t bcg_capture_id(hipStream_t stream) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  unsigned long long id = 0;
  if (hipStreamGetCaptureInfo(stream, &status, &id) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return status == hipStreamCaptureStatusActive ? static_cast<int64_t>(id) : 0;
}

// plan: of bcg_gemm_mid_plan for the same sizes, or any other tile and split.  epi: 0 store (+ bias), 1 silu(gate) * up of N / 2 features from w's first
// row on, their up rows `inter` rows behind, into rows of `c` that are `inter` apart, 2 residual + product (residual may be c).  x_scale [M],
// w_scale [N]: not null for e4m3 operands (epi 0 and 2).  Pointers 16-byte aligned, rows contiguous; ws and counters as
// bcg_gemm_mid_parts says.
BCG_API int bcg_gemm_mid(int plan, int epi, const void* x, const void* w, const float* x_scale, const float* w_scale, const void* bias,
                         const void* residual, void* c, void* ws, void* counters, int M, int N, int K, int inter, hipStream_t stream) {
  const bool f8 = x_scale != nullptr, gated = epi == EPI_SILU_MUL;
  const int bytes = f8 ? K : 2 * K, split = plan >> 8, tile = plan & 255;
  if (plan < 0 || tile >= N_TILES || M <= 0 || K <= 0 || bytes % 128 || N <= 0 || N % (gated ? 32 : 16) || N > 1 << 20) return -2;
  if (split < 1 || split > bytes / 128 || (split > 1 && (!ws || !counters)) || (f8 && !w_scale)) return -2;
  if (gated && (inter < N / 2 || inter % 16 || inter > 1 << 20)) return -2;
  if (static_cast<int64_t>(gated ? 2 * inter : N) * bytes >= 1ll << 31 || static_cast<int64_t>(M) * bytes >= 1ll << 31) return -2;
  const int bm = TILES[tile].mt * 16, bn = TILES[tile].nt * 16;
  const MidArgs a = {static_cast<const unsigned char*>(x), static_cast<const unsigned char*>(w), static_cast<const bf16_t*>(bias),
                     static_cast<const bf16_t*>(residual), static_cast<bf16_t*>(c), static_cast<float*>(ws), static_cast<int*>(counters),
                     x_scale, w_scale, M, N, inter, bytes / 128, (M + bm - 1) / bm, gated ? (N / 2 + bn / 2 - 1) / (bn / 2) : (N + bn - 1) / bn, split};
  if (static_cast<int64_t>(a.m_tiles) * a.n_tiles * split > 1 << 24 || static_cast<int64_t>(a.m_tiles) * a.n_tiles > 1 << 16) return -2;
  switch (epi) {
    case EPI_STORE: return f8 ? bcg_gemm_mid_fp8(tile, &a, stream) : launch<EPI_STORE, false>(tile, a, stream);
    case EPI_SILU_MUL: return f8 ? -2 : bcg_gemm_mid_gated(tile, &a, stream);
    case EPI_RESIDUAL:
      if (!residual) return -2;
      return f8 ? bcg_gemm_mid_fp8_residual(tile, &a, stream) : bcg_gemm_mid_residual(tile, &a, stream);
    default: return -2;
  }
}

// A projection and the activation behind it, bf16 without bias; plan: as bcg_gemm_mid's of the plain product, operands, ws and counters too.
// at > 0: c [M, at] = the first `at` columns of the product, other [M, N - at] = gelu (tanh form) of those behind; at < N, both multiples of 8.
// at == 0: c [M, N] = gelu of the product times columns 0 .. N - 1 of row tokens[m] of `other`, rows `ld` apart (a multiple of 8), tokens kept within
// 0 .. vocab - 1.
// The activation took a launch of 4.7 to 4.8 us at 64 rows; in here it adds 1.3 us to 64 x 18432 x 4096 (31.6 -> 32.9) and 0.4 to 64 x 256 x 2048 (6.7 -> 7.1).
// The product is rounded once, behind the activation.
BCG_API int bcg_gemm_mid_act(int plan, const void* x, const void* w, void* c, void* other, const int* tokens, void* ws, void* counters, int M, int N,
                             int K, int at, int ld, int vocab, hipStream_t stream) {
  const int split = plan >> 8, tile = plan & 255;
  if (plan < 0 || tile >= N_TILES || M <= 0 || K <= 0 || K % 64 || N <= 0 || N % 16 || N > 1 << 20 || !other) return -2;
  if (split < 1 || split > K / 64 || (split > 1 && (!ws || !counters))) return -2;
  if (at < 0 || at >= N || at % 8 || (at == 0 && (!tokens || vocab < 1 || ld < N || ld % 8))) return -2;
  if (2ll * N * K >= 1ll << 31 || 2ll * M * K >= 1ll << 31) return -2;
  const int bm = TILES[tile].mt * 16, bn = TILES[tile].nt * 16;
  MidArgs a = {};
  a.x = static_cast<const unsigned char*>(x), a.w = static_cast<const unsigned char*>(w), a.c = static_cast<bf16_t*>(c);
  a.ws = static_cast<float*>(ws), a.counters = static_cast<int*>(counters);
  a.M = M, a.N = N, a.blocks = K / 64, a.m_tiles = (M + bm - 1) / bm, a.n_tiles = (N + bn - 1) / bn, a.split = split, a.at = at;
  if (static_cast<int64_t>(a.m_tiles) * a.n_tiles * split > 1 << 24 || static_cast<int64_t>(a.m_tiles) * a.n_tiles > 1 << 16) return -2;
  if (at > 0) {
    a.tail = static_cast<bf16_t*>(other);
    return bcg_gemm_mid_tail_gelu(tile, &a, stream);
  }
  a.table = static_cast<const bf16_t*>(other), a.tokens = tokens, a.table_ld = ld, a.vocab = vocab;
  return bcg_gemm_mid_gelu_table(tile, &a, stream);
}
