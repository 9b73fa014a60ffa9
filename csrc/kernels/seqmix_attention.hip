// Multi-map (differential) causal GQA attention over a paged KV cache, fp32 scores and softmax.
//
//   head h, map m:  a_m = softmax(scale q_m K_m^T) V      (every map over the SAME values)
//   o = a_0 - lam a_1   (maps = 2;  maps = 1: a_0),   o <- o / sqrt(mean(o^2) + eps) * out_scale
//
// Cache of one layer run: K [NB, G, BS, maps dim], V [NB, G, vdim, BS] logically.  With `swz`
// (maps dim a multiple of 4) a (page, KV head) slab is stored fragment-major, so that the 64
// lanes of one MFMA operand load read 512 contiguous bytes instead of 64 scattered 8-byte pieces:
//   K slab [maps dim / 4][BS][4]  (4 features of one key, key after key, feature group after group)
//   V slab [BS / 4][vdim][4]      (4 keys of one value feature, feature after feature, key group after group)
// BS is a multiple of 16.
//
// prefill_kernel: a work tile is <= 64 query rows of one sequence (4 waves x 16 rows) for one
// query head.  Per 16 keys a wave computes S^T = K Q^T (keys x queries) with 16 x 16 MFMAs, so
// the C registers of S^T are already the B operand (keys x queries) of O^T = V^T P^T: no
// shuffle between the two products; softmax statistics are per query = per lane column
// (reduced over the 4 lane groups).  K / V^T fragments are read straight from the cache
// (a lane's share of an operand is 4 consecutive elements of one cache row).
//
// The bf16 instance for heads up to 64 / 128 wide takes 32 keys per iteration and prefetches
// the next iteration's K fragments in registers.
//
// prefill_staged_kernel: the same tiles for exact shapes with 16-token pages, K and V through LDS.
//
// decode_mfma_kernel: single-token rows.  The 16 MFMA columns hold the query heads that share
// one KV head (GQA packing), so the cache is read once per KV head; one wave per 128-key split.
// decode_merge_kernel merges the splits and applies the map combination + head norm.
//
// decode_pair_kernel: single-token rows of exact shapes with 16-token pages, a workgroup per (row, KV head x column group),
// or for each of a few parts of one.
//
// Optional, for one-map heads: a sliding window (a query at position i sees keys j with
// i - j < window) or a chunk mask (position i sees j <= i of its own chunk, floor(i / chunk) ==
// floor(j / chunk), chunks counted from position 0), and a per-head sink, a learned logit that takes part in the softmax denominator
// only (no key, no value, not scaled).  The key loop starts at the window's (chunk's) first 16-key
// tile; decode splits are counted from the window's (chunk's) first split.  A window may keep the
// sequence's first `keep` keys (KEEP instances): every query sees them at their true positions.  The
// key loop then walks the tiles of the kept keys, jumps to the window's first tile and goes on; decode
// splits are those that hold kept keys, then the window's.
//
// Optional score shape (SHAPED instances, one-map heads): the scaled score s becomes cap tanh(s / cap)
// (cap > 0), then slope_h (i - j) is taken off (slopes non-null).  Both act on fp32 scores.
#include <algorithm>

#include "seqmix_common.h"

namespace {

constexpr int SPLIT_KEYS = 128;
constexpr int PLAIN = 0, SHAPED = 1, KEEP = 2;   // loop forms: as is / capped or biased scores / kept first keys
constexpr float MAX_FLOOR = -1.0e30f;   // running maxima start finite: a tile may be hidden as a whole
constexpr float LOG2E = 1.4426950408889634f;

struct AttnArgs {
  const void* q;            // [T, H, maps dim]
  const void* k_cache;
  const void* v_cache;
  const int* block_tables;  // [B, max_blocks]
  const int* q_start;       // [B + 1] (prefill)
  const int* seq_lens;      // [B]
  const int* work;          // prefill: tiles [n, 3] {seq, row0, row_end}; decode: items [n, 2] {row, seq} or null
  void* out;                // [T, H vdim]
  float* ws;                // decode partials
  int max_blocks, H, G, maps, dim, vdim, BS, num_blocks, n_splits;
  float scale, lam, head_eps, out_scale;
  int vec_k, vec_v;         // rows of K / V^T are aligned for 4-element vector loads
  int window;               // > 0: keys below position - window + 1 are hidden
  int keep;                 // > 0 (with a window): keys below `keep` stay visible (KEEP instances)
  int chunk;                // > 0: keys below position - position % chunk are hidden (chunks count from position 0)
  const float* sink;        // [H] or null
  float softcap;            // > 0: scaled scores are capped, cap tanh(s / cap)   (SHAPED instances)
  const float* slopes;      // [H] or null: slope_h (i - j) is taken off the score (SHAPED instances)
  int swz;                  // fragment-major slabs (see the top of the file)
  PartRule rule;            // decode by pairs
  int n_items;
  int* counters;            // [rule.extra] zeros, left zero
};

// Maximum / sum over the four lanes that share a column (lanes col, col + 16, col + 32, col + 48): register swaps, no LDS
// round trip.
__device__ __forceinline__ float column_max(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float column_sum(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Two neighbouring 16-deep operands in one 32-deep product (bf16): the lanes' 4 + 4 elements of both operands pair up the
// same way, so the order of k inside the instruction is free.
__device__ __forceinline__ f32x4 mma32(s16x4 a0, s16x4 a1, s16x4 b0, s16x4 b1, f32x4 c) {
  typedef short s16x8 __attribute__((ext_vector_type(8)));
  const s16x8 a = __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7), b = __builtin_shufflevector(b0, b1, 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mma32(f32x4 a0, f32x4 a1, f32x4 b0, f32x4 b1, f32x4 c) { return mma16(a1, b1, mma16(a0, b0, c)); }

// The product of two rows of N operands, of which the first n_used hold something (the others are zero): every product of one
// depth, an odd last operand beside zeros.  The depths must not meet on one accumulator: a 16x16x16 product that takes
// the result of a 16x16x32 one (or the other way round) as its accumulator needs three wait states between the
// two, which hipcc does not insert when the registers are exactly the same -- it counts on the forwarding that
// two products of one form have.  Without them the sums are wrong (gfx950, ROCm 7.2: 0, 1 and 2 states wrong in half of the
// elements, 3 and more right); with the loads of two maps between them it showed at two 48-wide maps and not at one.
template <typename T, int N, typename FA, typename FB>
__device__ __forceinline__ f32x4 mma_row(int n_used, FA a, FB b) {
  f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < N; i += 2)
    if (i < n_used) {
      if (i + 1 < N) c = mma32(a(i), a(i + 1), b(i), b(i + 1), c);
      else c = mma32(a(i), zero_frag<T>(), b(i), zero_frag<T>(), c);
    }
  return c;
}

// First key that a query at position `pos` sees: the window's or the chunk's first, else 0.
__device__ __forceinline__ int first_key(const AttnArgs& a, int pos) {
  if (a.window > 0) return max(0, pos - a.window + 1);
  if (a.chunk > 0) return pos - pos % a.chunk;
  return 0;
}

// Decode splits of a row whose window starts at key `lo`: split i covers the keys of the absolute split
// `split_abs` -- first those that hold kept keys, then the window's.
__device__ __forceinline__ int keep_splits(const AttnArgs& a) { return (a.keep + SPLIT_KEYS - 1) / SPLIT_KEYS; }
__device__ __forceinline__ int split_abs_of(const AttnArgs& a, int lo, int split) {
  const int nk = keep_splits(a);
  return split < nk ? split : max(lo / SPLIT_KEYS, nk) + split - nk;
}
__device__ __forceinline__ int split_count(const AttnArgs& a, int lo, int ctx) {
  const int nk = keep_splits(a), total = (ctx + SPLIT_KEYS - 1) / SPLIT_KEYS;
  return total <= nk ? total : nk + total - max(lo / SPLIT_KEYS, nk);
}

// The key loop shared by both kernels: keys [k_begin, k_last] of one sequence for the 16 query
// columns of a wave (column = a query row of one head, or a query head of one token).
//   limit      per lane: the last key its column may see;  limit_min: the smallest over the wave
//   lo         per lane: the first key its column may see;  lo_max: the largest over the wave
//   KT         16-key tiles per iteration (one softmax update and one rescale per iteration)
//   PF         this iteration's V^T fragments are loaded before its QK^T products and the next
//              iteration's K fragments right after them (loads fly under the MFMAs and the softmax)
//   FULL       whole, aligned fragments only (no branch around any load)
//   MODE       SHAPED: scores are capped / biased: pos = the position of the lane's column, slope = its head's
//              slope times log2 e.  KEEP: keys below `keep` stay visible; once they are passed the loop
//              jumps to the tile at k_win (a multiple of 16)
// Everything that does not depend on the lane stays scalar: the page lookup and the slab base go
// to SGPRs, a lane adds a 32-bit offset that is fixed for the whole loop.  Scores are kept in the
// log2 domain (scale * log2 e folded into one multiply, v_exp_f32 directly).
template <typename T, int KC, int VT, int KT, bool PF, bool FULL, int EXACT, int NM, int MODE>
__device__ __forceinline__ void attend_range(const AttnArgs& a_, int g, const typename Elem<T>::frag (&qf)[NM][KC],
                                             int limit, int limit_min, int lo, int lo_max, int k_begin, int k_last,
                                             const int* __restrict__ table, f32x4 (&acc)[NM][VT], float (&mx)[NM],
                                             float (&den)[NM], int pos = 0, float slope = 0.f, int keep = 0,
                                             int k_win = 0) {
  typedef typename Elem<T>::frag F;
  // EXACT (1 or 2 = the number of maps): dim = 16 KC, vdim = 16 VT, 16-token pages, fragment-major slabs -- every guard
  // below is a compile-time constant, fragment offsets are immediates, the loop body is straight-line
  struct Shape {
    const AttnArgs& r;
    int maps, dim, vdim, swz, BS, G, max_blocks, num_blocks, vec_k, vec_v;
    float scale;
    const void *k_cache, *v_cache;
  };
  const Shape a{a_, EXACT ? EXACT : a_.maps, EXACT ? 16 * KC : a_.dim, EXACT ? 16 * VT : a_.vdim, EXACT ? 1 : a_.swz, EXACT ? 16 : a_.BS, a_.G,
                a_.max_blocks, a_.num_blocks, EXACT ? 1 : a_.vec_k, EXACT ? 1 : a_.vec_v, a_.scale, a_.k_cache, a_.v_cache};
  const int lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4;
  const int KD = a.maps * a.dim;
  const int kc = EXACT ? KC : (a.dim + 15) >> 4, vt = EXACT ? VT : (a.vdim + 15) >> 4;
  const bool vec_k = a.vec_k && (a.dim & 3) == 0;
  const float sc = a.scale * 1.4426950408889634f;
  // capped scores: cap tanh(s / cap) = cap - 2 cap / (exp(2 s / cap) + 1), in the log2 domain
  const float cap = MODE == SHAPED ? a_.softcap : 0.f;
  const float cap2 = cap * LOG2E, arg2 = cap > 0.f ? 2.0f * LOG2E * a.scale / cap : 0.f;
  auto shape_score = [&](float dot, int key, bool capped) {
    float v = dot * sc;
    if (capped) {
      if constexpr (sizeof(T) == 2) v = cap2 - 2.0f * cap2 * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(dot * arg2) + 1.0f);
      else v = cap2 * tanhf(dot * a.scale / cap);
    }
    return v - slope * static_cast<float>(pos - key);
  };
  // offsets inside a (page, KV head) slab = one lane offset (fixed for the whole loop) + a
  // wave-uniform offset per fragment; the slab base and the tile's key offset are uniform too
  const uint32_t k_lane = a.swz ? (grp * a.BS + col) * 4 : col * KD + 4 * grp;
  const uint32_t v_lane = a.swz ? (grp * a.vdim + col) * 4 : col * a.BS + 4 * grp;
  auto k_uni = [&](int m, int c) { return a.swz ? ((m * a.dim + 16 * c) >> 2) * a.BS * 4 : m * a.dim + 16 * c; };
  auto v_uni = [&](int t) { return a.swz ? 16 * t * 4 : 16 * t * a.BS; };
  const int k_mul = a.swz ? 4 : KD, v_mul = a.swz ? a.vdim : 1;   // slab offset per key of the tile's first key
  const T* kc_base = static_cast<const T*>(a.k_cache);
  const T* vc_base = static_cast<const T*>(a.v_cache);
  const size_t k_slab = static_cast<size_t>(a.BS) * KD, v_slab = static_cast<size_t>(a.BS) * a.vdim;

  // A cursor walks the sequence in 16-key tiles: page index + key offset in the page, stepped
  // without a division (BS is a multiple of 16).  Tiles past the sequence read some valid page:
  // every one of their keys is masked.
  struct Cursor { int p, o; };
  auto step = [&](Cursor& c) {
    c.o += 16;
    if (c.o >= a.BS) { c.o = 0; ++c.p; }
  };
  auto place = [&](Cursor& c, int key) {
    c.p = key / a.BS;
    c.o = key - c.p * a.BS;
  };
  // first key of the iteration behind the one at `key0`; KEEP: past the kept keys, on to the window
  auto next_key = [&](int key0) {
    const int n = key0 + 16 * KT;
    if constexpr (MODE == KEEP) return (n >= keep && n < k_win) ? k_win : n;
    else return n;
  };
  auto slab_base = [&](const Cursor& c) {
    int page = table[min(c.p, a.max_blocks - 1)];
    page = (page < 0 || page >= a.num_blocks) ? 0 : page;
    return static_cast<size_t>(page) * a.G + g;
  };
  auto load_k = [&](Cursor& c, F (&kf)[KT][NM][KC]) {
#pragma unroll
    for (int u = 0; u < KT; ++u) {
      const T* kp = kc_base + slab_base(c) * k_slab + c.o * k_mul;
      step(c);
#pragma unroll
      for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int c2 = 0; c2 < KC; ++c2)
          kf[u][m][c2] = (m < a.maps && c2 < kc) ? load_frag_t<T, FULL>(kp + k_uni(m, c2) + k_lane, a.dim - (16 * c2 + 4 * grp), vec_k)
                                                 : zero_frag<T>();
    }
  };

  Cursor k_cur, v_cur;
  place(k_cur, k_begin);
  v_cur = k_cur;
  F kf[KT][NM][KC];
  if (PF) load_k(k_cur, kf);
  for (int key0 = k_begin, key_next; key0 <= k_last; key0 = key_next) {
    key_next = next_key(key0);
    const T* vps[KT];
#pragma unroll
    for (int u = 0; u < KT; ++u) {
      vps[u] = vc_base + slab_base(v_cur) * v_slab + v_cur.o * v_mul;
      step(v_cur);
    }
    if constexpr (MODE == KEEP) {
      if (key_next != key0 + 16 * KT) {   // (wave-uniform) the jump
        place(v_cur, key_next);
        if (PF) place(k_cur, key_next);
      }
    }
    F vf[PF ? KT : 1][PF ? VT : 1];
    auto load_v = [&](int u, int t) {
      return (t < vt && 16 * t + col < a.vdim) ? load_frag_t<T, FULL>(vps[u] + v_uni(t) + v_lane, 4, a.vec_v) : zero_frag<T>();
    };
    if constexpr (PF) {
#pragma unroll
      for (int u = 0; u < KT; ++u)
#pragma unroll
        for (int t = 0; t < VT; ++t) vf[u][t] = load_v(u, t);
    } else {
      load_k(k_cur, kf);
      if constexpr (MODE == KEEP) {
        if (key_next != key0 + 16 * KT) place(k_cur, key_next);
      }
    }
    // ---- S^T = K Q^T ----
    f32x4 s[KT][NM];
#pragma unroll
    for (int u = 0; u < KT; ++u)
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        s[u][m] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (m < a.maps) s[u][m] = mma_row<T, KC>(kc, [&](int c) { return kf[u][m][c]; }, [&](int c) { return qf[m][c]; });
      }
    // the K fragments are spent: the next iteration's go into the same registers, under the
    // softmax and the second product
    if (PF && key_next <= k_last) load_k(k_cur, kf);
    // ---- online softmax per query column; lane holds keys key0 + 16 u + 4 grp + i ----
    const bool masked = key0 + 16 * KT - 1 > limit_min || key0 < lo_max;   // (wave-uniform) some key of the iteration is hidden
    // (opaque per iteration: one loop body, not one per combination of uniform conditions)
    float cap_now = cap;
    if constexpr (MODE == SHAPED) asm volatile("" : "+v"(cap_now));
    const bool capped = cap_now > 0.f;
    F pf[KT][NM];
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      if (m >= a.maps) {
#pragma unroll
        for (int u = 0; u < KT; ++u) pf[u][m] = zero_frag<T>();
        continue;
      }
      float v[KT][4], bm = -INFINITY;
#pragma unroll
      for (int u = 0; u < KT; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = key0 + 16 * u + 4 * grp + i;
          if constexpr (MODE == SHAPED) v[u][i] = shape_score(s[u][m][i], key, capped);
          else v[u][i] = s[u][m][i] * sc;
          if (masked && (key > limit || (key < lo && !(MODE == KEEP && key < keep)))) v[u][i] = -INFINITY;
          bm = fmaxf(bm, v[u][i]);
        }
      const float m_new = fmaxf(mx[m], column_max(bm));     // finite: the running maximum starts finite
      float ps = 0.f;
#pragma unroll
      for (int u = 0; u < KT; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v[u][i] = __builtin_amdgcn_exp2f(v[u][i] - m_new);
          ps += v[u][i];
        }
      if (__any(m_new > mx[m])) {                           // (wave-uniform) the running maximum moved
        const float alpha = __builtin_amdgcn_exp2f(mx[m] - m_new);
        den[m] *= alpha;
#pragma unroll
        for (int t = 0; t < VT; ++t)
          if (t < vt) acc[m][t] *= alpha;
      }
      den[m] += ps;
      mx[m] = m_new;
#pragma unroll
      for (int u = 0; u < KT; ++u) pf[u][m] = Elem<T>::pack(v[u][0], v[u][1], v[u][2], v[u][3]);
    }
    // ---- O^T += V^T P^T ----
    static_assert(KT <= 2, "one 32-deep product per 32 keys");
#pragma unroll
    for (int t = 0; t < VT; ++t)
      if (t < vt) {
        F x[KT];
#pragma unroll
        for (int u = 0; u < KT; ++u) {
          if constexpr (PF) x[u] = vf[u][t]; else x[u] = load_v(u, t);
        }
#pragma unroll
        for (int m = 0; m < NM; ++m)
          if (m < a.maps) {
            if constexpr (KT == 2) acc[m][t] = mma32(x[0], x[1], pf[0][m], pf[1][m], acc[m][t]);
            else acc[m][t] = mma16(x[0], pf[0][m], acc[m][t]);
          }
      }
  }
#pragma unroll
  for (int m = 0; m < NM; ++m) den[m] = column_sum(den[m]);
}

template <typename T, int KC, int VT, int KT, bool PF, bool FULL, int OCC, int EXACT = 0, int NM = 2, int MODE = PLAIN>
__global__ __launch_bounds__(256, OCC) void prefill_kernel(AttnArgs a) {
  typedef typename Elem<T>::frag F;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, grp = lane >> 4;
  const int h = blockIdx.y, g = h / (a.H / a.G);
  const int seq = a.work[3 * blockIdx.x], row0 = a.work[3 * blockIdx.x + 1] + 16 * wave, row_end = a.work[3 * blockIdx.x + 2];
  if (row0 >= row_end) return;
  const int ctx = a.seq_lens[seq], q_end = a.q_start[seq + 1];
  const int n_rows = min(16, row_end - row0);
  const int row = row0 + min(col, n_rows - 1);             // columns past the tile repeat its last row (never stored)
  const int pos = ctx - (q_end - row);                     // position of this lane's query column
  const int pos_min = ctx - (q_end - row0), pos_max = pos_min + n_rows - 1;
  const int KD = a.maps * a.dim;
  const int kc = (a.dim + 15) >> 4, vt = (a.vdim + 15) >> 4;
  const bool vec_k = a.vec_k && (a.dim & 3) == 0;
  const T* qrow = static_cast<const T*>(a.q) + (static_cast<size_t>(row) * a.H + h) * KD;

  F qf[NM][KC];
#pragma unroll
  for (int m = 0; m < NM; ++m)
#pragma unroll
    for (int c = 0; c < KC; ++c) {
      const int f = 16 * c + 4 * grp;
      qf[m][c] = (m < a.maps && c < kc) ? load_frag_t<T, FULL>(qrow + m * a.dim + f, a.dim - f, vec_k) : zero_frag<T>();
    }
  f32x4 acc[NM][VT];
#pragma unroll
  for (int m = 0; m < NM; ++m)
#pragma unroll
    for (int t = 0; t < VT; ++t) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float mx[NM], den[NM];
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    mx[m] = MAX_FLOOR;
    den[m] = 0.f;
  }
  if (a.sink != nullptr) {   // the sink starts the softmax: weight 1 at its own logit
    mx[0] = a.sink[h] * LOG2E;
    den[0] = grp == 0 ? 1.0f : 0.0f;   // (a column's denominator is summed over its lanes at the end)
  }
  const int lo = first_key(a, pos), lo_max = first_key(a, pos_max);   // (both masks: the first key grows with the position)
  const int k_win = first_key(a, pos_min) & ~15, k_begin = MODE == KEEP ? 0 : k_win;
  const float slope = MODE == SHAPED && a.slopes != nullptr ? a.slopes[h] * LOG2E : 0.f;
  attend_range<T, KC, VT, KT, PF, FULL, EXACT, NM, MODE>(a, g, qf, pos, pos_min, lo, lo_max, k_begin, pos_max,
                                        a.block_tables + static_cast<size_t>(seq) * a.max_blocks, acc, mx, den, pos, slope,
                                        a.keep, k_win);
  // ---- combine the maps, unit norm over the head's value features, store ----
  const float i0 = 1.0f / den[0];
  float i1 = 0.f;
  if constexpr (NM > 1) {
    if (a.maps > 1) i1 = a.lam / den[1];
  }
  float ss = 0.f;
#pragma unroll
  for (int t = 0; t < VT; ++t)
    if (t < vt) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float o = acc[0][t][i] * i0;
        if constexpr (NM > 1) {
          if (a.maps > 1) o -= acc[1][t][i] * i1;
        }
        acc[0][t][i] = o;
        ss += o * o;   // rows >= vdim are zero (their V^T fragments were zero)
      }
    }
  ss = column_sum(ss);
  const float r = (a.head_eps >= 0.f ? 1.0f / sqrtf(ss / a.vdim + a.head_eps) : 1.0f) * a.out_scale;
  if (col < n_rows) {
    T* orow = static_cast<T*>(a.out) + (static_cast<size_t>(row) * a.H + h) * a.vdim;
#pragma unroll
    for (int t = 0; t < VT; ++t)
      if (t < vt) {
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[0][t][i] *= r;
        const int e = 16 * t + 4 * grp;
        if (EXACT) {   // whole tiles, aligned rows
          *reinterpret_cast<F*>(orow + e) = Elem<T>::pack(acc[0][t][0], acc[0][t][1], acc[0][t][2], acc[0][t][3]);
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (e + i < a.vdim) orow[e + i] = Elem<T>::st(acc[0][t][i]);
        }
      }
  }
}

// Prefill tiles of exact shapes (bf16, 16-token pages, fragment-major slabs), the pages staged through LDS.
//
// What bounded the form above: each of its waves loads every K / V fragment for 16 query rows alone and waits for it,
// with registers for one block in flight.  Here the 4 waves of a tile read one copy: a chunk of 32 keys is two pages,
// each a contiguous run of K and of V, copied as it lies (16 bytes per thread and access; the next chunk is in flight
// in registers while this one is multiplied, the page numbers one chunk further ahead; two buffers, one barrier per
// chunk).  The fragments come from LDS at the offsets they have in the slab, the 4-key rows of V moved apart by 128
// bytes so that the lane groups read different banks.  All waves walk the tile's key range; a wave skips chunks that
// hold no key it sees.  The tile list is walked as it comes, the heads of a tile side by side: the engine lists the tiles with the
// most keys first, so the launch ends on short ones (backwards, on the longest: 149, 170, 36.6 and 30 us of the four below).
// Measured, 8 prompts of 1000 tokens: two 64-wide maps over 128-wide values, 16 heads: 226 us (one load per wave, 16-deep
// products) -> 190 (32-deep products, column statistics by register swaps) -> 127 here; 32 latent heads of 192 / 128:
// 379 -> 313 -> 162; 3 prompts of 700, 16 latent heads: 63 -> 35, 16 heads of 128 with a window: 52 -> 43 -> 28.  Two heads'
// waves on one copy (512 threads) measured the same at the large sizes and 41 against 36 us at the small one.  What is left: LDS
// reads (20 KB per 16 rows and chunk, 75 of the 162 us if alone) and softmax arithmetic, at 3 waves per SIMD.
template <int KC, int VT, int NM, int MODE>
__global__ __launch_bounds__(256, NM * (KC + 2 * VT) <= 24 ? 4 : KC + VT <= 24 ? 3 : 2) void prefill_staged_kernel(AttnArgs a) {
  typedef s16x4 F;
  constexpr int DIM = 16 * KC, VD = 16 * VT, KD = NM * DIM, TH = 256;
  constexpr int UNITS = 4 * (KD + VD), NU = (UNITS + TH - 1) / TH;   // 16-byte units of a chunk, and per thread
  constexpr int VROW = VD / 2 + 8, BUF = 4 * KD + 8 * VROW;          // LDS: the 4-key rows of V 128 bytes apart in banks
  __shared__ __attribute__((aligned(16))) f32x4 chunk_lds[2 * BUF];  // twice K page 0, K page 1, V page 0, V page 1
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, grp = lane >> 4;
  const int h = blockIdx.x % a.H, g = h / (a.H / a.G);
  const int* item = a.work + 3 * (blockIdx.x / a.H);
  const int seq = item[0], first = item[1], row_end = item[2];
  if (first >= row_end) return;   // (the whole workgroup) an entry without rows: its sequence and row need not exist
  const int row0 = first + 16 * wave;
  const bool active = row0 < row_end;
  const int ctx = a.seq_lens[seq], q_end = a.q_start[seq + 1];
  const int n_rows = active ? min(16, row_end - row0) : 1;
  const int row = (active ? row0 : first) + min(col, n_rows - 1);   // columns past the tile repeat its last row (never stored)
  const int pos = ctx - (q_end - row);
  const int pos_min = ctx - (q_end - (active ? row0 : first)), pos_max = pos_min + n_rows - 1;
  const int pos_first = ctx - (q_end - first), pos_last = ctx - (q_end - (row_end - 1));
  const bf16_t* qrow = static_cast<const bf16_t*>(a.q) + (static_cast<size_t>(row) * a.H + h) * KD;
  F qf[NM][KC];
#pragma unroll
  for (int m = 0; m < NM; ++m)
#pragma unroll
    for (int c = 0; c < KC; ++c) qf[m][c] = *reinterpret_cast<const F*>(qrow + m * DIM + 16 * c + 4 * grp);
  f32x4 acc[NM][VT];
  float mx[NM], den[NM];
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    mx[m] = MAX_FLOOR;
    den[m] = 0.f;
#pragma unroll
    for (int t = 0; t < VT; ++t) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  if (a.sink != nullptr) {   // the sink starts the softmax: weight 1 at its own logit
    mx[0] = a.sink[h] * LOG2E;
    den[0] = grp == 0 ? 1.0f : 0.0f;
  }
  const int lo = first_key(a, pos), lo_min = first_key(a, pos_min), lo_max = first_key(a, pos_max);
  const int k_win = first_key(a, pos_first) & ~15, k_begin = MODE == KEEP ? 0 : k_win, keep = MODE == KEEP ? a.keep : 0;
  const float sc = a.scale * LOG2E;
  const float slope = MODE == SHAPED && a.slopes != nullptr ? a.slopes[h] * LOG2E : 0.f;
  const float cap = MODE == SHAPED ? a.softcap : 0.f;
  const float cap2 = cap * LOG2E, arg2 = cap > 0.f ? 2.0f * LOG2E * a.scale / cap : 0.f;
  auto next_key = [&](int key0) {   // KEEP: past the kept keys, on to the window
    const int n = key0 + 32;
    if constexpr (MODE == KEEP) return (n >= keep && n < k_win) ? k_win : n;
    else return n;
  };

  const int* table = a.block_tables + static_cast<size_t>(seq) * a.max_blocks;
  const int last_page = min((ctx - 1) >> 4, a.max_blocks - 1);
  auto page_of = [&](int p) {   // past the sequence: its last page again, every key of it is masked
    const int page = table[min(p, last_page)];
    return static_cast<size_t>((page < 0 || page >= a.num_blocks) ? 0 : page) * a.G + g;
  };
  typedef f32x4 Unit __attribute__((aligned(8)));   // (one 16-byte load all the same: global loads need 4-byte alignment)
  f32x4 stage[NU];   // (the threads past the end of a chunk repeat its last unit)
  auto fetch = [&](size_t s0, size_t s1) {
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int u = min(tid + i * TH, UNITS - 1);
      const bool isv = u >= 4 * KD;
      const int w = isv ? VD : KD, r = isv ? u - 4 * KD : u, second = r >= 2 * w;
      const Unit* base = static_cast<const Unit*>(isv ? a.v_cache : a.k_cache);
      stage[i] = base[(second ? s1 : s0) * (2 * w) + (r - second * 2 * w)];
    }
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int u = min(tid + i * TH, UNITS - 1), v = u - 4 * KD;
      chunk_lds[buf * BUF + (v < 0 ? u : 4 * KD + v + v / (VD / 2) * 8)] = stage[i];
    }
  };

  int key0 = k_begin, nxt = next_key(k_begin);
  fetch(page_of(key0 >> 4), page_of((key0 >> 4) + 1));
  put(0);
  fetch(page_of(nxt >> 4), page_of((nxt >> 4) + 1));
  size_t p0 = page_of(next_key(nxt) >> 4), p1 = page_of((next_key(nxt) >> 4) + 1);   // the pages two chunks ahead
  __syncthreads();
  for (int buf = 0; key0 <= pos_last; buf ^= 1) {
    if (active && key0 <= pos_max && (key0 + 31 >= lo_min || key0 < keep)) {   // (wave-uniform) some key is seen
      const bf16_t* ks = reinterpret_cast<const bf16_t*>(chunk_lds + buf * BUF);
      const bf16_t* vs = ks + 32 * KD;
      f32x4 sm[2][NM];
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int m = 0; m < NM; ++m) {
          sm[u][m] = mma_row<bf16_t, KC>(
              KC, [&](int c) { return *reinterpret_cast<const F*>(ks + u * 16 * KD + ((m * DIM + 16 * c) / 4 * 16 + grp * 16 + col) * 4); },
              [&](int c) { return qf[m][c]; });
        }
      const bool masked = key0 + 31 > pos_min || key0 < lo_max;
      float cap_now = cap;
      if constexpr (MODE == SHAPED) asm volatile("" : "+v"(cap_now));
      const bool capped = cap_now > 0.f;
      F pf[2][NM];
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        float v[2][4], bm = -INFINITY;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int key = key0 + 16 * u + 4 * grp + i;
            if constexpr (MODE == SHAPED) {
              float x = sm[u][m][i] * sc;
              if (capped) x = cap2 - 2.0f * cap2 * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(sm[u][m][i] * arg2) + 1.0f);
              v[u][i] = x - slope * static_cast<float>(pos - key);
            } else {
              v[u][i] = sm[u][m][i] * sc;
            }
            if (masked && (key > pos || (key < lo && !(MODE == KEEP && key < keep)))) v[u][i] = -INFINITY;
            bm = fmaxf(bm, v[u][i]);
          }
        const float m_new = fmaxf(mx[m], column_max(bm));
        float ps = 0.f;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            v[u][i] = __builtin_amdgcn_exp2f(v[u][i] - m_new);
            ps += v[u][i];
          }
        if (__any(m_new > mx[m])) {
          const float alpha = __builtin_amdgcn_exp2f(mx[m] - m_new);
          den[m] *= alpha;
#pragma unroll
          for (int t = 0; t < VT; ++t) acc[m][t] *= alpha;
        }
        den[m] += ps;
        mx[m] = m_new;
#pragma unroll
        for (int u = 0; u < 2; ++u) pf[u][m] = Elem<bf16_t>::pack(v[u][0], v[u][1], v[u][2], v[u][3]);
      }
#pragma unroll
      for (int t = 0; t < VT; ++t) {
        const F x0 = *reinterpret_cast<const F*>(vs + grp * 8 * VROW + (16 * t + col) * 4);
        const F x1 = *reinterpret_cast<const F*>(vs + (4 + grp) * 8 * VROW + (16 * t + col) * 4);
#pragma unroll
        for (int m = 0; m < NM; ++m) acc[m][t] = mma32(x0, x1, pf[0][m], pf[1][m], acc[m][t]);
      }
    }
    if (nxt <= pos_last) put(buf ^ 1);   // (its readers passed the barrier of the chunk before)
    key0 = nxt;
    nxt = next_key(nxt);
    if (nxt <= pos_last) {
      fetch(p0, p1);
      const int n2 = next_key(nxt);
      p0 = page_of(n2 >> 4);
      p1 = page_of((n2 >> 4) + 1);
    }
    __syncthreads();
  }
  if (!active) return;
  float o_den[NM];
#pragma unroll
  for (int m = 0; m < NM; ++m) o_den[m] = (m == 0 ? 1.0f : a.lam) / column_sum(den[m]);
  float ss = 0.f;
#pragma unroll
  for (int t = 0; t < VT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float o = acc[0][t][i] * o_den[0];
      if constexpr (NM > 1) o -= acc[1][t][i] * o_den[1];
      acc[0][t][i] = o;
      ss += o * o;
    }
  ss = column_sum(ss);
  const float r = (a.head_eps >= 0.f ? 1.0f / sqrtf(ss / VD + a.head_eps) : 1.0f) * a.out_scale;
  if (col < n_rows) {
    bf16_t* orow = static_cast<bf16_t*>(a.out) + (static_cast<size_t>(row) * a.H + h) * VD;
#pragma unroll
    for (int t = 0; t < VT; ++t)
      *reinterpret_cast<F*>(orow + 16 * t + 4 * grp) = Elem<bf16_t>::pack(acc[0][t][0] * r, acc[0][t][1] * r, acc[0][t][2] * r, acc[0][t][3] * r);
  }
}

// what the copies of whole pages need: one page is a chunk's half, caches on 8 bytes like every 4-element fragment; and what its
// one-dimensional launch holds: fewer than 2^32 threads
inline bool staged_layout(const AttnArgs& a, int n_tiles) {
  return a.swz && a.BS == 16 && static_cast<int64_t>(n_tiles) * a.H < (1 << 24) && ((reinterpret_cast<uintptr_t>(a.k_cache) | reinterpret_cast<uintptr_t>(a.v_cache)) & 7) == 0;
}

template <int KC, int VT, int NM, int MODE>
int launch_staged(const AttnArgs& a, int n_tiles, hipStream_t s) {
  prefill_staged_kernel<KC, VT, NM, MODE><<<n_tiles * a.H, 256, 0, s>>>(a);
  return BCG_CHECK_LAUNCH();
}

// Single-token rows, the query heads of one KV head packed into the 16 MFMA columns: column c is
// head g (H / G) + 16 cg + c of the same token, so K and V^T are read once per KV head.  One wave
// per (item, KV head x column group, SPLIT_KEYS-key split); partials as the merge kernel reads them
// (running maxima in the log2 domain of `attend_range`).
template <typename T, int KC, int VT, int KT, bool PF, bool FULL, int OCC, int EXACT = 0, int NM = 2, int MODE = PLAIN>
__global__ __launch_bounds__(64, OCC) void decode_mfma_kernel(AttnArgs a) {
  typedef typename Elem<T>::frag F;
  const int lane = threadIdx.x, col = lane & 15, grp = lane >> 4;
  const int per = a.H / a.G;
  const int g = blockIdx.x % a.G, cg = blockIdx.x / a.G;
  const int split = blockIdx.y, item = blockIdx.z;
  const int row = a.work ? a.work[2 * item] : item, seq = a.work ? a.work[2 * item + 1] : item;
  const int ctx = a.seq_lens[seq];
  const int lo = first_key(a, ctx - 1);                             // first visible key
  const int split_abs = MODE == KEEP ? split_abs_of(a, lo, split) : lo / SPLIT_KEYS + split;   // splits count from the window's first
  int k_end = min(ctx, (split_abs + 1) * SPLIT_KEYS);
  const int k_win = max(split_abs * SPLIT_KEYS, lo & ~15);
  int k_begin = k_win;
  if constexpr (MODE == KEEP) {
    if (split_abs * SPLIT_KEYS < a.keep) k_begin = split_abs * SPLIT_KEYS;   // the split holds kept keys ...
    if (lo >= k_end) k_end = min(k_end, a.keep);                             // ... and none of the window's
  }
  if (k_begin >= k_end) return;
  const bool col_ok = 16 * cg + col < per;
  const int h = g * per + min(16 * cg + col, per - 1);
  const int KD = a.maps * a.dim;
  const int kc = (a.dim + 15) >> 4, vt = (a.vdim + 15) >> 4;
  const bool vec_k = a.vec_k && (a.dim & 3) == 0;
  const T* qrow = static_cast<const T*>(a.q) + (static_cast<size_t>(row) * a.H + h) * KD;
  F qf[NM][KC];
#pragma unroll
  for (int m = 0; m < NM; ++m)
#pragma unroll
    for (int c = 0; c < KC; ++c) {
      const int f = 16 * c + 4 * grp;
      qf[m][c] = (m < a.maps && c < kc) ? load_frag_t<T, FULL>(qrow + m * a.dim + f, a.dim - f, vec_k) : zero_frag<T>();
    }
  f32x4 acc[NM][VT];
#pragma unroll
  for (int m = 0; m < NM; ++m)
#pragma unroll
    for (int t = 0; t < VT; ++t) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float mx[NM], den[NM];
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    mx[m] = MAX_FLOOR;
    den[m] = 0.f;
  }
  const float slope = MODE == SHAPED && a.slopes != nullptr ? a.slopes[h] * LOG2E : 0.f;
  attend_range<T, KC, VT, KT, PF, FULL, EXACT, NM, MODE>(a, g, qf, k_end - 1, k_end - 1, lo, lo, k_begin, k_end - 1,
                                        a.block_tables + static_cast<size_t>(seq) * a.max_blocks, acc, mx, den, ctx - 1, slope,
                                        a.keep, k_win);
  if (!col_ok) return;
  float* w = a.ws + ((static_cast<size_t>(item) * a.H + h) * a.n_splits + split) * (2 * a.maps + a.maps * a.vdim);
#pragma unroll
  for (int m = 0; m < NM; ++m)
    if (grp == 0 && m < a.maps) {
      w[m] = mx[m];
      w[a.maps + m] = den[m];
    }
#pragma unroll
  for (int m = 0; m < NM; ++m)
#pragma unroll
    for (int t = 0; t < VT; ++t)
      if (m < a.maps && t < vt) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int e = 16 * t + 4 * grp + i;
          if (e < a.vdim) w[2 * a.maps + m * a.vdim + e] = acc[m][t][i];
        }
      }
}

// The same rows for exact shapes (bf16, 16-token pages, fragment-major slabs), a workgroup per part of an (item, KV head x column group) pair.
//
// Its waves take the pair's 32-key chunks in turns and meet in LDS.  A page's slab is contiguous, so K and V come by LDS-DMA, 1 KB
// of a slab in one piece, each wave's into a chunk of its own, fetched again as soon as its fragments are in registers (V's 4-key groups with
// their 128-byte halves swapped in every other one, so that the lane groups of a fragment read differ in banks).  They are merged, combined and
// normed here, those of a row in several parts by the part that arrives last.  Against a wave per split of 128 keys and the merge of all splits it saves a
// launch and the splits' way through memory, and its loads are 16 bytes a lane instead of 8.  What bounds it: memory from some 256 pairs on (4.8 to
// 5.1 TB/s), below that a CU's intake and the chain of table, fetch, sums and merge.
// us, splits and merge -> this (spread lengths): two 64-wide maps over 128-wide values, 32 heads on 8, 64 rows of 1000 74 -> 54, 1 of 40 11 -> 6.2, 2 of 2000 24.1 ->
// 15.5 (8 parts), 200 of 500 114 -> 86; 16 latent heads of 192 / 128 behind a window of 512, 64 rows 14.8 -> 11.4, 1 row of 500 11.0 -> 9.0; 32 heads on 8 of
// 128 behind a window of 512, 16 rows 14.7 -> 11.1.  Two waves from 1025 pairs on, whose prologues hide behind more pairs: 200 rows of 40 tokens, 8 KV
// heads, two maps 25 -> 18 (splits 21), one 128-wide map 21 -> 15 (16.7); of 500 tokens 80.4, 80 and 76, 80.
template <int KC, int VT, int NM, int MODE, int NW>
__global__ __launch_bounds__(64 * NW, NM * KC + VT > 24 ? 1 : 2) void decode_pair_kernel(AttnArgs a) {
  typedef s16x4 F;
  constexpr int DIM = 16 * KC, VD = 16 * VT, KD = NM * DIM;
  constexpr int KB = KD * 32, VB = VD * 32, KP = KB / 1024, VP = VB / 1024, RING = 2 * (KB + VB);   // bytes of a page of K and of V, KB, of a wave's chunk
  static_assert(KB % 1024 == 0 && VB % 1024 == 0, "whole pieces");
  static_assert((VD * 17 + 64) * 4 <= RING && 16 * VD * 4 <= NW * RING, "the parts of the waves lie where the chunks were");
  static_assert((16 + 16 * 32 + 17 * 16 + 16 * VD) * 4 <= NW * RING, "and the factors of up to 16 parts of a row and their sums");
  constexpr int SWAP = VD % 32 == 0 ? 128 : 0;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[NW * RING];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), col = lane & 15, grp = lane >> 4;
  const int per = a.H / a.G, columns = a.G * ((per + 15) / 16);
  const Place place = place_of(a.rule, blockIdx.x, a.n_items * columns);
  const int at_item = place.at / columns, column = place.at - at_item * columns, g = column % a.G, cg = column / a.G;
  // (constant address space: scalar loads, whose wait is not one for the fetches)
  typedef const __attribute__((address_space(4))) int* Ints;
  auto ints = [](const int* p) { return reinterpret_cast<Ints>(reinterpret_cast<uintptr_t>(p)); };
  // a row's chunks: those that hold kept keys come before the window's, which begin with the page of the window's first key (a page in front of it may hold
  // what are no numbers, and a weight of zero does not take these out)
  const int keep = MODE == KEEP ? a.keep : 0, kept = (keep + 31) / 32;
  auto win_of = [&](int ctx_) { return max(first_key(a, ctx_ - 1) & ~15, 32 * kept); };
  auto chunks_of = [&](int ctx_) { return ctx_ > 0 ? min(kept, (ctx_ + 31) / 32) + max(0, ctx_ - win_of(ctx_) + 31) / 32 : 0; };
  auto chunks = [&](int i) { return chunks_of(a.seq_lens[a.work ? a.work[2 * i + 1] : i]); };
  Share sh{place.own ? at_item : -1, 0, 1, 0};
  if (__builtin_expect(a.rule.extra > 0 && (!place.own || a.rule.each == 0 ||
                                            chunks_of(ints(a.seq_lens)[a.work ? ints(a.work)[2 * at_item + 1] : at_item]) > a.rule.one), 0)) {
    sh = find_share(a.rule, a.n_items, columns, sh.row, at_item, chunks);
    if (sh.row < 0) return;   // (the whole workgroup)
  }
  const int item = sh.row, part = sh.part, parts = sh.n;
  const int row = a.work ? ints(a.work)[2 * item] : item, seq = a.work ? ints(a.work)[2 * item + 1] : item;
  const int ctx = ints(a.seq_lens)[seq], pos = ctx - 1;
  const Ints table = ints(a.block_tables) + static_cast<size_t>(seq) * a.max_blocks;
  const int lo = first_key(a, pos), win = win_of(ctx);
  const int all = chunks_of(ctx), begin = part * all / parts, end = (part + 1) * all / parts;   // this part's chunks
  const int last_page = min(max(ctx - 1, 0) / 16, a.max_blocks - 1);
  auto key_of = [&](int j) { return MODE != KEEP || j >= kept ? win + 32 * (j - kept) : 32 * j; };
  auto page_of = [&](int p) {   // past the sequence: its last page again, every key of it is masked
    const int page = table[min(p, last_page)];
    return static_cast<size_t>((page < 0 || page >= a.num_blocks) ? 0 : page) * a.G + g;
  };
  const uint32_t ring = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem)) + w * RING;
  auto dma = [&](uint32_t off, const unsigned char* base, uint32_t to) {   // (s_nop: the wait state of an LDS load behind a scalar write of m0)
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "s"(to) : "memory", "m0");
  };
  const unsigned char* kc_base = static_cast<const unsigned char*>(a.k_cache);
  const unsigned char* vc_base = static_cast<const unsigned char*>(a.v_cache);
  auto fetch_k = [&](size_t s0, size_t s1) {
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int i = 0; i < KP; ++i) dma(i * 1024 + lane * 16, kc_base + (e ? s1 : s0) * KB, ring + e * KB + i * 1024);
  };
  auto fetch_v = [&](size_t s0, size_t s1) {
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int i = 0; i < VP; ++i) {
        const uint32_t at = i * 1024 + lane * 16;
        dma(SWAP ? at ^ ((at / (VD * 8) & 1) * SWAP) : at, vc_base + (e ? s1 : s0) * VB, ring + 2 * KB + e * VB + i * 1024);
      }
  };
  size_t s0 = 0, s1 = 0;
  auto look = [&](int j) {
    const int p = key_of(j) / 16;
    s0 = page_of(p);
    s1 = page_of(p + 1);
  };
  const int h = g * per + min(16 * cg + col, per - 1);
  const bf16_t* qrow = static_cast<const bf16_t*>(a.q) + (static_cast<size_t>(row) * a.H + h) * KD;
  F qf[NM][KC];
#pragma unroll
  for (int m = 0; m < NM; ++m)
#pragma unroll
    for (int c = 0; c < KC; ++c) qf[m][c] = *reinterpret_cast<const F*>(qrow + m * DIM + 16 * c + 4 * grp);
  const float slope = MODE == SHAPED && a.slopes != nullptr ? a.slopes[h] * LOG2E : 0.f;
  // (all of these are here before the first fetch: a wait for them behind it would be one for the chunk)
#pragma unroll
  for (int m = 0; m < NM; ++m)
#pragma unroll
    for (int c = 0; c < KC; ++c) asm volatile("" : "+v"(qf[m][c]));
  if (begin + w < end) {
    look(begin + w);
    fetch_k(s0, s1);
    fetch_v(s0, s1);
  }
  f32x4 acc[NM][VT];
  float mx[NM], den[NM];
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    mx[m] = MAX_FLOOR;
    den[m] = 0.f;
#pragma unroll
    for (int t = 0; t < VT; ++t) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const float sc = a.scale * LOG2E;
  const float cap = MODE == SHAPED ? a.softcap : 0.f;
  const float cap2 = cap * LOG2E, arg2 = cap > 0.f ? 2.0f * LOG2E * a.scale / cap : 0.f;
  const bf16_t* ks = reinterpret_cast<const bf16_t*>(smem + w * RING);
  const unsigned char* vs = smem + w * RING + 2 * KB;
  const uint32_t v_lane = grp * VD * 8 + ((col * 8) ^ ((grp & 1) * SWAP));   // (a feature tile is 128 bytes: tiles alternate between the halves)

  for (int j = begin + w; j < end; j += NW) {
    const bool more = j + NW < end;
    if (more) look(j + NW);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * VP) : "memory");   // all but this chunk's V
    F kf[2][NM][KC];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int c = 0; c < KC; ++c) kf[u][m][c] = *reinterpret_cast<const F*>(ks + u * 16 * KD + ((m * DIM + 16 * c) / 4 * 16 + grp * 16 + col) * 4);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (more) {
      fetch_k(s0, s1);
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * KP) : "memory");   // all but the next chunk's K
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    F vf[2][VT];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int t = 0; t < VT; ++t) {
        const uint32_t at = SWAP ? (v_lane ^ (t % 2 * 128)) + t / 2 * 256 : v_lane + t * 128;
        vf[u][t] = *reinterpret_cast<const F*>(vs + u * VB + at);
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (more) fetch_v(s0, s1);
    f32x4 sm[2][NM];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int m = 0; m < NM; ++m) sm[u][m] = mma_row<bf16_t, KC>(KC, [&](int c) { return kf[u][m][c]; }, [&](int c) { return qf[m][c]; });
    const int key0 = key_of(j);
    const bool masked = key0 + 31 > pos || key0 < lo;
    float cap_now = cap;
    if constexpr (MODE == SHAPED) asm volatile("" : "+v"(cap_now));
    const bool capped = cap_now > 0.f;
    F pf[2][NM];
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      float v[2][4], bm = -INFINITY;
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = key0 + 16 * u + 4 * grp + i;
          if constexpr (MODE == SHAPED) {
            float y = sm[u][m][i] * sc;
            if (capped) y = cap2 - 2.0f * cap2 * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(sm[u][m][i] * arg2) + 1.0f);
            v[u][i] = y - slope * static_cast<float>(pos - key);
          } else {
            v[u][i] = sm[u][m][i] * sc;
          }
          if (masked && (key > pos || (key < lo && !(MODE == KEEP && key < keep)))) v[u][i] = -INFINITY;
          bm = fmaxf(bm, v[u][i]);
        }
      const float m_new = fmaxf(mx[m], column_max(bm));
      float ps = 0.f;
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v[u][i] = __builtin_amdgcn_exp2f(v[u][i] - m_new);
          ps += v[u][i];
        }
      if (__any(m_new > mx[m])) {
        const float alpha = __builtin_amdgcn_exp2f(mx[m] - m_new);
        den[m] *= alpha;
#pragma unroll
        for (int t = 0; t < VT; ++t) acc[m][t] *= alpha;
      }
      den[m] += ps;
      mx[m] = m_new;
#pragma unroll
      for (int u = 0; u < 2; ++u) pf[u][m] = Elem<bf16_t>::pack(v[u][0], v[u][1], v[u][2], v[u][3]);
    }
#pragma unroll
    for (int t = 0; t < VT; ++t)
#pragma unroll
      for (int m = 0; m < NM; ++m) acc[m][t] = mma32(vf[0][t], vf[1][t], pf[0][m], pf[1][m], acc[m][t]);
  }

  // ---- the waves' parts meet, map after map (every fetch has landed: the last chunk of a wave waits for all of its own)
  constexpr int TH = 64 * NW, N_OUT = 16 * VD / TH;    // elements of the heads' outputs per thread
  float* ml = reinterpret_cast<float*>(smem);          // [NW][2][16]
  float* fac = ml + NW * 32;                           // [NW][16] factors of the waves' parts, [16] of their sum
  float* po = fac + NW * 32;                           // [NW][VD][17]
  const int heads = min(16, per - 16 * cg), h0 = g * per + 16 * cg;
  float res[N_OUT];                                    // element tid + TH i: head, value feature
  // where a part of a cut row lies: [2 extra] slots of [16][NM][VD] numerators, then [16][2][NM] maxima and denominators; the first part behind the others
  constexpr int SLOT = 16 * (NM * VD + 2 * NM);
  auto slot_at = [&](int p) { return static_cast<uint32_t>((p > 0 ? (sh.first + p - 1) * columns : a.rule.extra + sh.first * columns) + column) * SLOT; };
  auto slot_ml = [&](int p, int hh, int den, int m) { return a.ws + slot_at(p) + 16 * NM * VD + (2 * hh + den) * NM + m; };
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    const float d = column_sum(den[m]);
    __syncthreads();
    if (grp == 0) {
      ml[w * 32 + col] = mx[m];
      ml[w * 32 + 16 + col] = d;
    }
#pragma unroll
    for (int t = 0; t < VT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) po[(w * VD + 16 * t + 4 * grp + i) * 17 + col] = acc[m][t][i];
    __syncthreads();
    if (tid < 16) {
      const bool sinks = m == 0 && parts == 1 && a.sink != nullptr && tid < heads;
      const float sink = sinks ? a.sink[h0 + tid] * LOG2E : MAX_FLOOR;
      float mm = sink;
#pragma unroll
      for (int x = 0; x < NW; ++x) mm = fmaxf(mm, ml[x * 32 + tid]);
      float ll = sinks ? exp2f(sink - mm) : 0.f;
#pragma unroll
      for (int x = 0; x < NW; ++x) {
        const float f = exp2f(ml[x * 32 + tid] - mm);
        fac[x * 16 + tid] = f;
        ll += ml[x * 32 + 16 + tid] * f;
      }
      fac[NW * 16 + tid] = (m == 0 ? 1.0f : -a.lam) / ll;
      if (parts > 1 && tid < heads) {
        store_through(slot_ml(part, tid, 0, m), mm);
        store_through(slot_ml(part, tid, 1, m), ll);
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N_OUT; ++i) {
      const int idx = tid + TH * i, hh = idx / VD, e = idx % VD;
      if (hh >= heads) break;
      float oo = 0.f;
#pragma unroll
      for (int x = 0; x < NW; ++x) oo += po[(x * VD + e) * 17 + hh] * fac[x * 16 + hh];
      if (parts > 1) {
        store_through(a.ws + slot_at(part) + (hh * NM + m) * VD + e, oo);
      } else {
        const float c = fac[NW * 16 + hh];
        res[i] = m == 0 ? oo * c : res[i] + oo * c;
      }
    }
  }
  if (parts > 1) {   // the last part of a cut row to arrive adds them up, always in their order
    if (!last_of(a.counters + sh.first * columns + column, parts, reinterpret_cast<int*>(smem))) return;
    const __amdgpu_buffer_rsrc_t rp = __builtin_amdgcn_make_buffer_rsrc(a.ws, 0, 2u * a.rule.extra * SLOT * 4, 0x00020000);
    f32x4 v[8];
    auto load_eight = [&](int p0, int m, int idx) {    // (past the last part: that one again, which is not added; past the heads: zeros)
#pragma unroll
      for (int j = 0; j < 8; ++j)
        v[j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                             rp, idx < heads * VD ? (slot_at(min(p0 + j, parts - 1)) + (idx / VD * NM + m) * VD + idx % VD) * 4 : 0xfffffff0u, 0, 16 /*sc1*/));
    };
    float* pml = reinterpret_cast<float*>(smem) + 16;  // [16 parts][2][16]
    float* pf = pml + 16 * 32;                         // [16 parts][16], [16] of their sum
    float* sum = pf + 17 * 16;                         // [16][VD]
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      if (m > 0) __syncthreads();
      load_eight(0, m, 4 * tid);                       // (beside the maxima)
      for (int i = tid; i < parts * 32; i += TH)
        if ((i & 15) < heads) pml[i] = load_through(slot_ml(i >> 5, i & 15, (i >> 4) & 1, m));
      __syncthreads();
      if (tid < heads) {
        const bool sinks = m == 0 && a.sink != nullptr;
        const float sink = sinks ? a.sink[h0 + tid] * LOG2E : MAX_FLOOR;
        float mm = sink;
        for (int p = 0; p < parts; ++p) mm = fmaxf(mm, pml[p * 32 + tid]);
        float ll = sinks ? exp2f(sink - mm) : 0.f;
        for (int p = 0; p < parts; ++p) {
          const float f = exp2f(pml[p * 32 + tid] - mm);
          pf[p * 16 + tid] = f;
          ll += pml[p * 32 + 16 + tid] * f;
        }
        pf[16 * 16 + tid] = (m == 0 ? 1.0f : -a.lam) / ll;
      }
      __syncthreads();
      for (int idx = 4 * tid; idx < heads * VD; idx += 4 * TH) {
        const int hh = idx / VD;
        f32x4 oo = {0.f, 0.f, 0.f, 0.f};
        for (int p0 = 0; p0 < parts; p0 += 8) {
          if (p0 > 0 || idx != 4 * tid) load_eight(p0, m, idx);
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (p0 + j < parts) oo += v[j] * pf[(p0 + j) * 16 + hh];
        }
        oo *= pf[16 * 16 + hh];
        f32x4* to = reinterpret_cast<f32x4*>(sum + idx);
        *to = m == 0 ? oo : *to + oo;
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N_OUT; ++i) res[i] = tid + TH * i < heads * VD ? sum[tid + TH * i] : 0.f;
  }
  bf16_t* rows = static_cast<bf16_t*>(a.out) + (static_cast<size_t>(row) * a.H + h0) * VD;
  if (a.head_eps < 0.f) {   // no norm
#pragma unroll
    for (int i = 0; i < N_OUT; ++i) {
      if ((tid + TH * i) / VD >= heads) break;
      rows[tid + TH * i] = f2bf(res[i] * a.out_scale);
    }
    return;
  }
  __syncthreads();
  float* out = reinterpret_cast<float*>(smem);         // [16][VD]
#pragma unroll
  for (int i = 0; i < N_OUT; ++i) {
    if ((tid + TH * i) / VD >= heads) break;
    out[tid + TH * i] = res[i];
  }
  __syncthreads();
  for (int hh = w; hh < heads; hh += NW) {
    float ss = 0.f;
    for (int e = lane; e < VD; e += 64) ss += out[hh * VD + e] * out[hh * VD + e];
    ss = wave_sum(ss);
    const float r = 1.0f / sqrtf(ss / VD + a.head_eps) * a.out_scale;
    for (int e = lane; e < VD; e += 64) rows[hh * VD + e] = f2bf(out[hh * VD + e] * r);
  }
}

// ws layout per (item, head, split): [maps] max, [maps] denominator, [maps][vdim] numerators.  A wave per head: the
// lanes take the splits' maxima and denominators side by side, then the splits' numerators, four in flight (a split after
// the other, each behind the load of its maximum, cost 20.5 us at 64 rows x 32 heads x 8 splits of two 128-wide maps;
// now 13.0).  VPL: value features per lane, two neighbours per access.
template <typename T, int VPL>
__global__ __launch_bounds__(64) void decode_merge_kernel(AttnArgs a) {
  const int lane = threadIdx.x, h = blockIdx.x, item = blockIdx.y;
  const int row = a.work ? a.work[2 * item] : item, seq = a.work ? a.work[2 * item + 1] : item;
  const int ctx = a.seq_lens[seq];
  const int n = min(a.n_splits, split_count(a, first_key(a, ctx - 1), ctx));
  const float sink = a.sink != nullptr ? a.sink[h] * LOG2E : MAX_FLOOR;
  const int stride = 2 * a.maps + a.maps * a.vdim;
  const float* w = a.ws + (static_cast<size_t>(item) * a.H + h) * a.n_splits * stride;
  const bool even = (a.vdim & 1) == 0;   // pairs of features are 8-byte aligned
  float o[VPL];
#pragma unroll
  for (int j = 0; j < VPL; ++j) o[j] = 0.f;
  for (int m = 0; m < a.maps; ++m) {
    float mx = m == 0 ? sink : MAX_FLOOR;
    for (int s = lane; s < n; s += 64) mx = fmaxf(mx, w[s * stride + m]);
    mx = wave_max(mx);
    float den = (m == 0 && a.sink != nullptr && lane == 0) ? exp2f(sink - mx) : 0.f, num[VPL];
#pragma unroll
    for (int j = 0; j < VPL; ++j) num[j] = 0.f;
    for (int s0 = 0; s0 < n; s0 += 64) {
      float fl = 0.f;   // (maxima are kept in the log2 domain)
      if (s0 + lane < n) {
        fl = exp2f(w[(s0 + lane) * stride + m] - mx);
        den += w[(s0 + lane) * stride + a.maps + m] * fl;
      }
      const float* v = w + s0 * stride + 2 * a.maps + m * a.vdim;
#pragma unroll 4
      for (int s = 0; s < min(64, n - s0); ++s) {
        const float f = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(fl), s));
#pragma unroll
        for (int j = 0; j < VPL; j += 2) {
          const int e = 2 * lane + 64 * j;
          if (even) {
            if (e < a.vdim) {
              const float2 x = *reinterpret_cast<const float2*>(v + s * stride + e);
              num[j] += x.x * f;
              num[j + 1] += x.y * f;
            }
          } else {
            if (e < a.vdim) num[j] += v[s * stride + e] * f;
            if (e + 1 < a.vdim) num[j + 1] += v[s * stride + e + 1] * f;
          }
        }
      }
    }
    const float c = (m == 0 ? 1.0f : -a.lam) / wave_sum(den);
#pragma unroll
    for (int j = 0; j < VPL; ++j) o[j] += num[j] * c;
  }
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < VPL; ++j) ss += o[j] * o[j];   // (features past vdim are zero)
  ss = wave_sum(ss);
  const float r = (a.head_eps >= 0.f ? 1.0f / sqrtf(ss / a.vdim + a.head_eps) : 1.0f) * a.out_scale;
  T* orow = static_cast<T*>(a.out) + (static_cast<size_t>(row) * a.H + h) * a.vdim;
#pragma unroll
  for (int j = 0; j < VPL; j += 2) {
    const int e = 2 * lane + 64 * j;
    if (e < a.vdim) orow[e] = Elem<T>::st(o[j] * r);
    if (e + 1 < a.vdim) orow[e + 1] = Elem<T>::st(o[j + 1] * r);
  }
}

// Exact one-map instances (bf16): X(KC, VT, keys tiles per iteration, workgroups per CU).
#define BCG_EXACT1_PLAIN(X) X(8, 8, 2, 2) X(4, 4, 2, 2) X(4, 8, 2, 2) X(2, 2, 2, 2) X(6, 6, 2, 2) X(6, 4, 2, 2) X(12, 8, 2, 2) \
                            X(12, 12, 2, 1) X(16, 16, 2, 1)
#define BCG_EXACT1_KEEP(X) X(8, 8, 2, 2) X(4, 4, 2, 2) X(4, 8, 2, 2) X(2, 2, 2, 2) X(6, 6, 2, 2) X(12, 12, 2, 1) X(16, 16, 2, 1)
#define BCG_EXACT1_SHAPED(X) X(8, 8, 2, 2) X(4, 4, 2, 2) X(2, 2, 2, 2) X(3, 3, 2, 2) X(6, 6, 2, 2) X(12, 12, 2, 1) X(16, 16, 2, 1)

// Heads whose scores are capped or biased, or whose window keeps first keys (one map).
template <typename T, int MODE>
int launch_prefill_mode(const AttnArgs& a, int n_tiles, bool full, hipStream_t s) {
  dim3 grid(n_tiles, a.H);
  if constexpr (sizeof(T) == 2) if (full && staged_layout(a, n_tiles)) {
#define BCG_X(KC_, VT_, KT_, OCC_)                                                               \
  if (a.dim == 16 * KC_ && a.vdim == 16 * VT_) {                                                 \
    return launch_staged<KC_, VT_, 1, MODE>(a, n_tiles, s);                                      \
  }
    if constexpr (MODE == SHAPED) { BCG_EXACT1_SHAPED(BCG_X) } else { BCG_EXACT1_KEEP(BCG_X) }
#undef BCG_X
  }
  if (a.dim <= 64 && a.vdim <= 128) prefill_kernel<T, 4, 8, 1, false, false, 1, 0, 1, MODE><<<grid, 256, 0, s>>>(a);
  else if (a.dim <= 256 && a.vdim <= 256) prefill_kernel<T, 16, 16, 1, false, false, 1, 0, 1, MODE><<<grid, 256, 0, s>>>(a);
  else prefill_kernel<T, 32, 32, 1, false, false, 1, 0, 1, MODE><<<grid, 256, 0, s>>>(a);
  return BCG_CHECK_LAUNCH();
}

template <typename T, int MODE>
void launch_decode_mode(const AttnArgs& a, dim3 grid, bool full, hipStream_t s) {
  if constexpr (sizeof(T) == 2) if (full && a.swz && a.BS == 16) {
#define BCG_X(KC_, VT_, KT_, OCC_)                                                               \
  if (a.dim == 16 * KC_ && a.vdim == 16 * VT_) {                                                 \
    decode_mfma_kernel<T, KC_, VT_, KT_, true, true, OCC_, 1, 1, MODE><<<grid, 64, 0, s>>>(a);   \
    return;                                                                                      \
  }
    if constexpr (MODE == SHAPED) { BCG_EXACT1_SHAPED(BCG_X) } else { BCG_EXACT1_KEEP(BCG_X) }
#undef BCG_X
  }
  if (a.dim <= 64 && a.vdim <= 128) decode_mfma_kernel<T, 4, 8, 1, false, false, 1, 0, 1, MODE><<<grid, 64, 0, s>>>(a);
  else if (a.dim <= 256 && a.vdim <= 256) decode_mfma_kernel<T, 16, 16, 1, false, false, 1, 0, 1, MODE><<<grid, 64, 0, s>>>(a);
  else decode_mfma_kernel<T, 32, 32, 1, false, false, 1, 0, 1, MODE><<<grid, 64, 0, s>>>(a);
}

template <typename T>
int launch_prefill(const AttnArgs& a, int n_tiles, int tile_rows, hipStream_t s) {
  dim3 grid(n_tiles, a.H);
  const bool small = a.dim <= 64 && a.vdim <= 128;
  const bool full = a.dim % 16 == 0 && a.vdim % 16 == 0 && a.vec_k && a.vec_v;   // whole, aligned fragments only
  if (tile_rows != 64) return -2;
  if (a.softcap > 0.f || a.slopes != nullptr) return launch_prefill_mode<T, SHAPED>(a, n_tiles, full, s);
  if (a.keep > 0) return launch_prefill_mode<T, KEEP>(a, n_tiles, full, s);
  if constexpr (sizeof(T) == 2) if (full && a.maps == 1 && staged_layout(a, n_tiles)) {   // one-map heads, exact shapes
#define BCG_X(KC_, VT_, KT_, OCC_)                                                               \
  if (a.dim == 16 * KC_ && a.vdim == 16 * VT_) {                                                 \
    return launch_staged<KC_, VT_, 1, PLAIN>(a, n_tiles, s);                                     \
  }
    BCG_EXACT1_PLAIN(BCG_X)
#undef BCG_X
    if (a.dim == 512 && a.vdim == 512) {   // (two chunks of it take 130 of the CU's 160 KiB: one workgroup per CU; that form is not built)
      prefill_kernel<T, 32, 32, 1, true, true, 1, 1, 1><<<grid, 256, 0, s>>>(a);
      return BCG_CHECK_LAUNCH();
    }
  }
  if constexpr (sizeof(T) == 2) if (small) {
    const bool exact = full && a.maps == 2 && staged_layout(a, n_tiles);
#define BCG_EXACT(KC_, VT_)                                                                      \
  if (exact && a.dim == 16 * KC_ && a.vdim == 16 * VT_) {                                        \
    return launch_staged<KC_, VT_, 2, PLAIN>(a, n_tiles, s);                                     \
  }
    BCG_EXACT(4, 8) BCG_EXACT(3, 6) BCG_EXACT(2, 4) BCG_EXACT(4, 4) BCG_EXACT(2, 2)
#undef BCG_EXACT
    if (full) prefill_kernel<T, 4, 8, 2, true, true, 2><<<grid, 256, 0, s>>>(a);
    else prefill_kernel<T, 4, 8, 2, true, false, 2><<<grid, 256, 0, s>>>(a);
    return BCG_CHECK_LAUNCH();
  }
  if (small) {
    if (full) prefill_kernel<T, 4, 8, 1, false, true, 2><<<grid, 256, 0, s>>>(a);
    else prefill_kernel<T, 4, 8, 1, false, false, 2><<<grid, 256, 0, s>>>(a);
  } else if (a.vdim > 256) {   // one map of more than 256 value features (a wide latent)
    prefill_kernel<T, 32, 32, 1, false, false, 1, 0, 1><<<grid, 256, 0, s>>>(a);
  } else if (a.dim <= 128) {   // (the branch-free form of the wide instance runs out of registers)
    prefill_kernel<T, 8, 16, 1, false, false, 1><<<grid, 256, 0, s>>>(a);
  } else if (a.dim <= 256) {   // one map of up to 256 key features (a latent plus a rotated part)
    prefill_kernel<T, 16, 16, 1, false, false, 1, 0, 1><<<grid, 256, 0, s>>>(a);
  } else {   // ... up to 512 (slow: the fragments of a row fill the register file)
    prefill_kernel<T, 32, 16, 1, false, false, 1, 0, 1><<<grid, 256, 0, s>>>(a);
  }
  return BCG_CHECK_LAUNCH();
}

template <typename T>
void launch_merge(const AttnArgs& a, int n_items, hipStream_t s) {
  if (a.vdim <= 128) decode_merge_kernel<T, 2><<<dim3(a.H, n_items), 64, 0, s>>>(a);
  else if (a.vdim <= 256) decode_merge_kernel<T, 4><<<dim3(a.H, n_items), 64, 0, s>>>(a);
  else decode_merge_kernel<T, 8><<<dim3(a.H, n_items), 64, 0, s>>>(a);
}

// Pairs of a decode step by a.rule (decode_pair_kernel); -2: not these heads.  n_items 0: only says whether.
int launch_pairs(const AttnArgs& a, hipStream_t s) {
  const int pairs = a.n_items * a.G * ((a.H / a.G + 15) / 16);
  const bool many = pairs + (a.rule.each == 0 ? a.rule.extra : 0) > 1024;   // (see decode_pair_kernel)
  auto run = [&](auto kernel4, auto kernel2) {
    if (a.n_items == 0) return 0;
    if (many) kernel2<<<pairs + a.rule.extra, 128, 0, s>>>(a);
    else kernel4<<<pairs + a.rule.extra, 256, 0, s>>>(a);
    return BCG_CHECK_LAUNCH();
  };
#define BCG_X(KC_, VT_, KT_, OCC_)                                                               \
  if constexpr ((KC_) % 2 == 0) if (a.dim == 16 * KC_ && a.vdim == 16 * VT_) return run(decode_pair_kernel<KC_, VT_, 1, BCG_MODE, 4>, decode_pair_kernel<KC_, VT_, 1, BCG_MODE, 2>);
  if (a.maps == 1 && (a.softcap > 0.f || a.slopes != nullptr)) {
#define BCG_MODE SHAPED
    BCG_EXACT1_SHAPED(BCG_X)
#undef BCG_MODE
    return -2;
  }
  if (a.maps == 1 && a.keep > 0) {
#define BCG_MODE KEEP
    BCG_EXACT1_KEEP(BCG_X)
#undef BCG_MODE
    return -2;
  }
  if (a.maps == 1) {
#define BCG_MODE PLAIN
    BCG_EXACT1_PLAIN(BCG_X)
#undef BCG_MODE
    return -2;
  }
#undef BCG_X
#define BCG_X(KC_, VT_) if (a.dim == 16 * KC_ && a.vdim == 16 * VT_) return run(decode_pair_kernel<KC_, VT_, 2, PLAIN, 4>, decode_pair_kernel<KC_, VT_, 2, PLAIN, 2>);
  BCG_X(4, 8) BCG_X(3, 6) BCG_X(2, 4) BCG_X(4, 4) BCG_X(2, 2)
#undef BCG_X
  return -2;
}

// Splits of 128 keys and their merge: fp32, heads or pages of other sizes, and of the exact sizes capped or sloped heads of 48 (a page of them is no whole number
// of KB) and caches that do not begin on 16 bytes, which the copies of decode_pair_kernel need.
// us, guarded instances in their place and this: 64 rows of 1000 tokens, heads of 48 capped, 16 on 4, 38.5, 20.1; caches off 16 bytes, 32 heads on 8 of 128 254, 65, two
// 64-wide maps over 128 84, 75, 16 latent heads of 192 / 128 behind a window of 512 60, 16.6 (on 16 bytes by pairs: 55 with the maps, 13).
template <typename T>
int launch_decode(const AttnArgs& a, int n_items, hipStream_t s) {
  const int per = a.H / a.G;
  dim3 grid(a.G * ((per + 15) / 16), a.n_splits, n_items);
  const bool full = a.dim % 16 == 0 && a.vdim % 16 == 0 && a.vec_k && a.vec_v;
  const bool shaped = a.softcap > 0.f || a.slopes != nullptr;
  bool done = shaped || a.keep > 0;
  if (shaped) launch_decode_mode<T, SHAPED>(a, grid, full, s);
  else if (done) launch_decode_mode<T, KEEP>(a, grid, full, s);
  if constexpr (sizeof(T) == 2) if (!done && full && a.maps == 1 && a.swz && a.BS == 16) {   // one-map heads, exact shapes
#define BCG_X(KC_, VT_, KT_, OCC_)                                                               \
  if (!done && a.dim == 16 * KC_ && a.vdim == 16 * VT_) {                                        \
    done = true;                                                                                 \
    decode_mfma_kernel<T, KC_, VT_, KT_, true, true, OCC_, 1, 1><<<grid, 64, 0, s>>>(a);         \
  }
    BCG_EXACT1_PLAIN(BCG_X)
    if (!done && a.dim == 512 && a.vdim == 512) {
      done = true;
      decode_mfma_kernel<T, 32, 32, 1, true, true, 1, 1, 1><<<grid, 64, 0, s>>>(a);
    }
#undef BCG_X
  }
  if constexpr (sizeof(T) == 2) if (!done && a.dim <= 64 && a.vdim <= 128) {
    done = true;
    const bool exact = full && a.maps == 2 && a.swz && a.BS == 16;
    bool hit = false;
#define BCG_EXACT(KC_, VT_)                                                                      \
  if (!hit && exact && a.dim == 16 * KC_ && a.vdim == 16 * VT_) {                                \
    hit = true;                                                                                  \
    decode_mfma_kernel<T, KC_, VT_, 2, true, true, 2, 2><<<grid, 64, 0, s>>>(a);                 \
  }
    BCG_EXACT(4, 8) BCG_EXACT(3, 6) BCG_EXACT(2, 4) BCG_EXACT(4, 4) BCG_EXACT(2, 2)
#undef BCG_EXACT
    if (hit) {
    } else
    if (full) decode_mfma_kernel<T, 4, 8, 2, true, true, 2><<<grid, 64, 0, s>>>(a);
    else decode_mfma_kernel<T, 4, 8, 2, true, false, 2><<<grid, 64, 0, s>>>(a);
  }
  if (done) {
  } else if (a.dim <= 64 && a.vdim <= 128) {
    if (full) decode_mfma_kernel<T, 4, 8, 1, false, true, 2><<<grid, 64, 0, s>>>(a);
    else decode_mfma_kernel<T, 4, 8, 1, false, false, 2><<<grid, 64, 0, s>>>(a);
  } else if (a.vdim > 256) {
    decode_mfma_kernel<T, 32, 32, 1, false, false, 1, 0, 1><<<grid, 64, 0, s>>>(a);
  } else if (a.dim <= 128) {
    decode_mfma_kernel<T, 8, 16, 1, false, false, 1><<<grid, 64, 0, s>>>(a);
  } else if (a.dim <= 256) {
    decode_mfma_kernel<T, 16, 16, 1, false, false, 1, 0, 1><<<grid, 64, 0, s>>>(a);
  } else {
    decode_mfma_kernel<T, 32, 16, 1, false, false, 1, 0, 1><<<grid, 64, 0, s>>>(a);
  }
  launch_merge<T>(a, n_items, s);
  return BCG_CHECK_LAUNCH();
}

}  // namespace

BCG_API int bcg_multimap_split_keys() { return SPLIT_KEYS; }

// mode 0: prefill tiles (work = tiles [n_work, 3]); mode 1: single-token items (work = [n_work, 2]
// {row, sequence}, or null: item i is row i of sequence i), n_splits the most splits of a row; mode 2: the same where bcg_multimap_pairs says
// so, with n_splits, one, each, ways and extra the rule by which several workgroups take a pair of a long row (PartRule; extra >= the parts beyond a pair's first
// that the rule can make: ways or pairs (n_splits - 1), each 0: the latter): ws 2 extra 16 (2 maps + maps vdim) floats, counters `extra` zeros, left zero.
BCG_API int bcg_multimap_attention(int mode, const void* q, const void* k_cache, const void* v_cache,
                                   const void* block_tables, int max_blocks, const void* q_start, const void* seq_lens,
                                   const void* work, int n_work, void* out, void* ws, int n_splits, int H, int G, int maps,
                                   int dim, int vdim, int BS, int num_blocks, float scale, float lam, float head_eps,
                                   float out_scale, int tile_rows, int is_f32, int window, int chunk, const void* sink,
                                   float softcap, const void* slopes, int keep, int one, int each, int ways, int extra, int* counters, void* stream) {
  if (n_work <= 0) return 0;
  if (keep < 0 || (keep > 0 && (window <= 0 || softcap != 0.f || slopes != nullptr))) return -2;
  if ((window > 0 || chunk > 0 || sink != nullptr || softcap != 0.f || slopes != nullptr) && maps != 1) return -2;
  if (window > 0 && chunk > 0) return -2;
  if (maps < 1 || maps > 2 || dim > (maps == 1 ? 512 : 128) || vdim > (maps == 1 ? 512 : 256) || BS % 16 || H % G || n_work > 65535 * 16) return -2;
  AttnArgs a;
  a.q = q; a.k_cache = k_cache; a.v_cache = v_cache;
  a.block_tables = static_cast<const int*>(block_tables); a.q_start = static_cast<const int*>(q_start);
  a.seq_lens = static_cast<const int*>(seq_lens); a.work = static_cast<const int*>(work);
  a.out = out; a.ws = static_cast<float*>(ws);
  a.max_blocks = max_blocks; a.H = H; a.G = G; a.maps = maps; a.dim = dim; a.vdim = vdim; a.BS = BS;
  a.num_blocks = num_blocks; a.n_splits = n_splits;
  a.scale = scale; a.lam = lam; a.head_eps = head_eps; a.out_scale = out_scale;
  a.vec_k = ((maps * dim) % 4 == 0) ? 1 : 0;
  a.vec_v = 1;  // BS % 16 == 0: every 4-key group of a V^T row is aligned
  a.swz = a.vec_k;
  a.window = window; a.keep = keep; a.chunk = chunk; a.sink = static_cast<const float*>(sink);
  a.softcap = softcap; a.slopes = static_cast<const float*>(slopes);
  hipStream_t s = static_cast<hipStream_t>(stream);
  a.n_items = n_work;
  a.rule = PartRule{n_splits, one, each, ways, extra};
  a.counters = counters;
  if (mode == 2) {
    const int64_t pairs = static_cast<int64_t>(n_work) * G * ((H / G + 15) / 16), most = pairs * (n_splits - 1);
    if (is_f32 || BS != 16 || !a.swz || n_splits < 1 || n_splits > 16 || H > 65535 || n_work > 65535 || pairs >= 1 << 30 || max_blocks < 1 || one < 0 || each < 0 ||
        extra < (each > 0 && most > ways ? ways : most) || extra > 1 << 16 || ways < 0 ||
        ((reinterpret_cast<uintptr_t>(k_cache) | reinterpret_cast<uintptr_t>(v_cache)) & 15) || (extra > 0 && (!ws || !counters)))
      return -2;
    return launch_pairs(a, s);
  }
  if (mode == 0) return is_f32 ? launch_prefill<float>(a, n_work, tile_rows, s) : launch_prefill<bf16_t>(a, n_work, tile_rows, s);
  if (n_splits < 1 || H > 65535 || n_splits > 65535 || n_work > 65535) return -2;
  return is_f32 ? launch_decode<float>(a, n_work, s) : launch_decode<bf16_t>(a, n_work, s);
}

// Whether mode 2 takes the decode steps of these heads (bf16, 16-token pages, caches on 16 bytes).
BCG_API int bcg_multimap_pairs(int maps, int dim, int vdim, int shaped, int keep) {
  AttnArgs a{};
  a.maps = maps, a.dim = dim, a.vdim = vdim, a.softcap = shaped ? 1.f : 0.f, a.keep = keep, a.H = a.G = 1;
  return (maps == 1 || maps == 2) && launch_pairs(a, nullptr) == 0;
}
