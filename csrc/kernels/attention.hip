// Paged GQA attention on MFMA (v_mfma_f32_16x16x32_bf16) for decode and prefill.
//
// "Swapped" formulation (cdna_hip_programming.md, Appendix B, fused attention):
//   S^T = K · Q^T      A = K rows straight from the paged cache (16 tokens x 32 dims),
//                      B = Q^T fragment held in registers for the whole loop;
//   O^T += V^T · P^T   A = V^T read from the *transposed* V cache ([hd][BS] per
//                      block-head), B = P^T built lane-locally from the S^T
//                      accumulators (no LDS, no shuffles).
// Every per-query quantity (running max m, sum l, rescale factor, O^T column)
// lives on lane column q = lane & 15: the online softmax needs two
// xor-shuffles per 32-token chunk and no data movement between the MFMAs.
//
// MFMA 16x16x32 bf16 lane maps (gfx950):
//   A[row = l&15][k = 8(l>>4)+j], B[k = 8(l>>4)+j][col = l&15], C[row = 4(l>>4)+i][col = l&15]
// Token permutation of a 32-token chunk (makes every V fragment ONE 16-byte load):
//   S^T tile u (u = 0,1), C row 4h+i  <->  chunk token 8h + 4u + i
//   so lane group h holds the scores of tokens 8h..8h+7, which is exactly the
//   k-slot order (h, j) <-> token 8h+j of the P^T / V^T operands; tokens 8h..8h+7
//   are 16 contiguous bytes of one V^T row (block h>>1, offset 8(h&1)).
//   K tiles load row r from token 8(r>>2) + 4u + (r&3) (a row gather: free).
//
// Decode: one workgroup per (sequence, kv head, 256-token split), or, where the batch has more
// of these than the chip holds, an even share of all chunks per wave (`decode_stream`); the
// G = n_q/n_kv query heads of the kv head share every K/V byte (GQA packing: 5 for Qwen3-14B);
// waves are combined through LDS and splits merged by a second kernel
// (flash-decoding).  Prefill: one workgroup per (64-query tile, query
// head), causal over cached prefix + new tokens, varlen via a tile table.

#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "common.h"

namespace {

constexpr int BS = 16;            // KV block size (tokens)
constexpr int DEC_WAVES = 4;
constexpr int CHUNK = 32;
constexpr float LOG2E = 1.4426950408889634f;
constexpr float RESCALE_LOG2 = 8.f;  // lazy online-softmax rescale threshold (log2 units)

// 2^x as the bare v_exp_f32.  exp2f() wraps it in a denormal range reduction (v_cmp +
// v_cndmask + v_ldexp around every exponential: ~3 extra VALU per score); softmax
// arguments are <= 0 here and a result below 2^-126 may flush to 0.
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Single-instruction maxima.  fmaxf() on MFMA results makes hipcc canonicalise every input
// first (one v_max_f32 x, x per score: 32 extra VALU per 64 MFMAs in the prefill loop); the
// scores here are never NaN, so the raw v_max3 / v_max forms are exact.
__device__ __forceinline__ float vmax3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
__device__ __forceinline__ float vmax(float a, float b) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
typedef float f32x2 __attribute__((ext_vector_type(2)));

struct KVGeom {
  const bf16_t* k;   // [L, NB, n_kv, BS, HD]
  const bf16_t* v;   // [L, NB, n_kv, HD, BS]
  int layer, num_blocks, n_kv;
};

template <int HD>
__device__ __forceinline__ size_t block_base(const KVGeom& g, int blk, int kvh) {
  return ((static_cast<size_t>(g.layer) * g.num_blocks + blk) * g.n_kv + kvh) * (BS * HD);
}

// A chunk's operands as loaded: bf16x8 (16 B) per fragment, or -- fp8 KV cache --
// the raw 8 e4m3fn bytes, widened to bf16 only right before their MFMA so the
// loads of the next chunk stay in flight (converting at load time would wait).
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <int HD, bool F8 = false>
struct Chunk {
  typedef typename std::conditional<F8, u32x2, bf16x8>::type E;
  E k[2][HD / 32];   // S^T A-operands, tile u, k-step kk
  E v[HD / 16];      // O^T A-operands, d-tile dt
};

__device__ __forceinline__ bf16x8 to_bf16x8(const bf16x8& x) { return x; }

__device__ __forceinline__ bf16x8 to_bf16x8(const u32x2& x) {  // 8 x e4m3fn -> 8 x bf16 (exact)
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const bf16x2 a = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(x[0], 1.f, false);
  const bf16x2 b = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(x[0], 1.f, true);
  const bf16x2 c = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(x[1], 1.f, false);
  const bf16x2 d = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(x[1], 1.f, true);
  return bf16x8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

// Issue every load of one 32-token chunk whose blocks are blk0/blk1.
template <int HD, bool F8 = false>
__device__ __forceinline__ void load_chunk(Chunk<HD, F8>& c, const KVGeom& g, int blk0, int blk1, int kvh,
                                           int lane) {
  typedef typename Chunk<HD, F8>::E E;
  typedef typename std::conditional<F8, uint8_t, bf16_t>::type T;  // cache element
  const T* kc = reinterpret_cast<const T*>(g.k);
  const T* vc = reinterpret_cast<const T*>(g.v);
  const int r = lane & 15, h = lane >> 4;
  const size_t b0 = block_base<HD>(g, blk0, kvh), b1 = block_base<HD>(g, blk1, kvh);
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int t = 8 * (r >> 2) + 4 * u + (r & 3);
    const T* krow = kc + (t < BS ? b0 : b1) + (t & (BS - 1)) * HD + 8 * h;
#pragma unroll
    for (int kk = 0; kk < HD / 32; ++kk) c.k[u][kk] = *reinterpret_cast<const E*>(krow + kk * 32);
  }
  const T* vb = vc + (h < 2 ? b0 : b1) + 8 * (h & 1);
#pragma unroll
  for (int dt = 0; dt < HD / 16; ++dt) c.v[dt] = *reinterpret_cast<const E*>(vb + (dt * 16 + r) * BS);
  // Keep all 16 loads of the chunk together: without this fence hipcc sinks the
  // V loads below the S^T MFMAs that wait for K, i.e. two serial HBM round trips.
  __builtin_amdgcn_sched_barrier(0);
}

// The K half / V half of load_chunk, for loops that reload a chunk's registers in place
// (K right after the S^T MFMAs consumed it, V after the P.V MFMAs).
template <int HD, bool F8 = false>
__device__ __forceinline__ void load_chunk_k(Chunk<HD, F8>& c, const KVGeom& g, int blk0, int blk1, int kvh,
                                             int lane) {
  typedef typename Chunk<HD, F8>::E E;
  typedef typename std::conditional<F8, uint8_t, bf16_t>::type T;
  const T* kc = reinterpret_cast<const T*>(g.k);
  const int r = lane & 15, h = lane >> 4;
  const size_t b0 = block_base<HD>(g, blk0, kvh), b1 = block_base<HD>(g, blk1, kvh);
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int t = 8 * (r >> 2) + 4 * u + (r & 3);
    const T* krow = kc + (t < BS ? b0 : b1) + (t & (BS - 1)) * HD + 8 * h;
#pragma unroll
    for (int kk = 0; kk < HD / 32; ++kk) c.k[u][kk] = *reinterpret_cast<const E*>(krow + kk * 32);
  }
}

template <int HD, bool F8 = false>
__device__ __forceinline__ void load_chunk_v(Chunk<HD, F8>& c, const KVGeom& g, int blk0, int blk1, int kvh,
                                             int lane) {
  typedef typename Chunk<HD, F8>::E E;
  typedef typename std::conditional<F8, uint8_t, bf16_t>::type T;
  const T* vc = reinterpret_cast<const T*>(g.v);
  const int r = lane & 15, h = lane >> 4;
  const T* vb = vc + block_base<HD>(g, h < 2 ? blk0 : blk1, kvh) + 8 * (h & 1);
#pragma unroll
  for (int dt = 0; dt < HD / 16; ++dt) c.v[dt] = *reinterpret_cast<const E*>(vb + (dt * 16 + r) * BS);
}

// Reductions over the 4 lane rows (h = lane >> 4) that share a query column:
// v_permlane16_swap (rows 0<->1, 2<->3) then v_permlane32_swap (0<->2, 1<->3),
// two VALU ops each instead of ds_bpermute round trips through the LDS
// crossbar (~100 cycles apiece, four of them in series per chunk).  Both
// halves of each swap are combined, so every lane gets identical bits.
__device__ __forceinline__ float rows_max(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = vmax(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return vmax(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

__device__ __forceinline__ float rows_sum(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Online-softmax update + O^T accumulation for one chunk starting at token t0.
// visible(t) decides masking (t = absolute token index); kv_end bounds V reads.
// MASKED = false: the caller guarantees every token of the chunk is visible to
// every column (wave-uniform), so the per-token mask and the V-tail zeroing
// (~60 VALU ops per chunk beside 16 MFMAs) are skipped.
template <int HD, typename Vis, bool MASKED = true, bool F8 = false, bool LAZY = true>
__device__ __forceinline__ void compute_chunk(const Chunk<HD, F8>& c, const bf16x8 (&bq)[HD / 32], int t0, int kv_end,
                                              Vis visible, float scale_log2, float& m, float& l,
                                              f32x4 (&o)[HD / 16], int lane) {
  const int h = lane >> 4;
  f32x4 s[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    s[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < HD / 32; ++kk)
      s[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(to_bf16x8(c.k[u][kk]), bq[kk], s[u], 0, 0, 0);
  }
  float p[8];
  float mx = -INFINITY;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int t = t0 + 8 * h + j;
    const float sv = s[j >> 2][j & 3];
    p[j] = (!MASKED || (t < kv_end && visible(t))) ? sv * scale_log2 : -INFINITY;
    mx = fmaxf(mx, p[j]);
  }
  mx = rows_max(mx);
  // Lazy rescale: the reference max m only moves when some column's chunk max
  // exceeds it by more than 2^RESCALE_LOG2 (then P <= 2^8 stays exact in fp32 /
  // bf16 and l cannot overflow over an 8k context).  Rescaling O is 32 VALU
  // multiplies plus the accumulator moves around them -- the kernels were
  // VALU-bound on it (14 VALU per MFMA, PMC); after the first chunks it is rare.
  if constexpr (LAZY) {
    if (__builtin_amdgcn_ballot_w64(mx > m + RESCALE_LOG2) != 0) {  // wave-uniform
      const float m_new = fmaxf(m, mx);
      const float alpha = m == -INFINITY ? 0.f : fast_exp2(m - m_new);
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < HD / 16; ++dt) o[dt] *= alpha;
      m = m_new;
    }
  }
  // eager (LAZY = false): rescale every chunk, O folded into the P.V loop below --
  // the branch-free form keeps fewer registers live (no spills at NT = 4)
  float alpha = 1.f;
  if constexpr (!LAZY) {
    const float m_new = fmaxf(m, mx);
    alpha = m == -INFINITY ? 0.f : fast_exp2(m - (m_new == -INFINITY ? 0.f : m_new));
    l *= alpha;
    m = m_new;
  }
  const float m_use = m == -INFINITY ? 0.f : m;
  float ps = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    p[j] = fast_exp2(p[j] - m_use);
    ps += p[j];
  }
  ps = rows_sum(ps);
  l += ps;
  bf16x8 bp;
#pragma unroll
  for (int j = 0; j < 8; ++j) bp[j] = static_cast<__bf16>(p[j]);
  // tokens past kv_end may hold stale (even non-finite) bytes: zero their V
  // with branch-free 32-bit masks (a divergent branch here splits the vmcnt waits)
  if constexpr (MASKED) {
    uint32_t keep[4];
#pragma unroll
    for (int j2 = 0; j2 < 4; ++j2) {
      const int t = t0 + 8 * h + 2 * j2;
      keep[j2] = (t < kv_end ? 0x0000ffffu : 0u) | (t + 1 < kv_end ? 0xffff0000u : 0u);
    }
#pragma unroll
    for (int dt = 0; dt < HD / 16; ++dt) {
      if constexpr (!LAZY) o[dt] *= alpha;
      u32x4 va = __builtin_bit_cast(u32x4, to_bf16x8(c.v[dt]));
#pragma unroll
      for (int j2 = 0; j2 < 4; ++j2) va[j2] &= keep[j2];
      o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, va), bp, o[dt], 0, 0, 0);
    }
  } else {
#pragma unroll
    for (int dt = 0; dt < HD / 16; ++dt) {
      if constexpr (!LAZY) o[dt] *= alpha;
      o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(to_bf16x8(c.v[dt]), bp, o[dt], 0, 0, 0);
    }
  }
}


// All NT query sub-tiles of a wave on one chunk that every row of every sub-tile sees in
// full (no mask), as ONE straight-line block: the S^T MFMAs of every sub-tile first, then
// each sub-tile's softmax (its VALU runs while the later sub-tiles' MFMAs are still in the
// pipe), then every P.V MFMA.  Split in two so the caller's loop can leave for the (rare,
// lazy: only when some column's running max moves by > 2^RESCALE_LOG2) rescale of O:
//   full_scores  S^T MFMAs, the next chunk's K reloaded in place, per-column chunk max;
//                returns whether any column needs a rescale (wave-uniform);
//   full_pv      P = exp2(S - m), l += rowsum(P), O^T += V^T P^T, next chunk's V reloaded.
// With the rescale (VALU on the O accumulators) inside the loop body, hipcc copied all
// 128 O accumulators AGPR -> VGPR at the top of EVERY chunk, taken or not (128
// v_accvgpr_read per 64 MFMAs at NT = 4); outside it, O stays in AGPRs.
template <int HD, int NT, bool F8, typename ReloadK>
__device__ __forceinline__ bool full_scores(Chunk<HD, F8>& c, const bf16x8 (&bq)[NT][HD / 32], float scale_log2,
                                            const float (&m)[NT], f32x2 (&t)[NT][4], float (&mx)[NT],
                                            ReloadK reload_k) {
  f32x4 s[NT][2];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      s[nt][u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < HD / 32; ++kk)
        s[nt][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(to_bf16x8(c.k[u][kk]), bq[nt][kk], s[nt][u], 0, 0, 0);
    }
  reload_k(c);  // next chunk's K into the registers the S^T MFMAs just read
  // every score is read from the MFMA result ONCE: t = S * scale - m (two per v_pk_fma_f32), its
  // column max decides the lazy rescale, and full_pv exponentiates t directly
  // (before the first chunk m = -inf: t is taken relative to 0 and the chunk always rescales)
  bool grow = false;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const bool first = m[nt] == -INFINITY;
    const float m_eff = first ? 0.f : m[nt];
    const f32x2 sc = {scale_log2, scale_log2}, mm = {m_eff, m_eff};
#pragma unroll
    for (int q = 0; q < 4; ++q)
      t[nt][q] = f32x2{s[nt][q >> 1][2 * (q & 1)], s[nt][q >> 1][2 * (q & 1) + 1]} * sc - mm;
    const float v = vmax3(vmax3(t[nt][0].x, t[nt][0].y, t[nt][1].x), vmax3(t[nt][1].y, t[nt][2].x, t[nt][2].y),
                          vmax(t[nt][3].x, t[nt][3].y));
    const float rel = rows_max(v);  // chunk max relative to the running max
    mx[nt] = rel + m_eff;
    grow |= first || rel > RESCALE_LOG2;
  }
  return __builtin_amdgcn_ballot_w64(grow) != 0;
}

template <int HD, int NT, bool F8, typename ReloadV>
__device__ __forceinline__ void full_pv(Chunk<HD, F8>& c, const f32x2 (&t)[NT][4], float (&l)[NT],
                                        f32x4 (&o)[NT][HD / 16], ReloadV reload_v) {
  bf16x8 bp[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    f32x2 p[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      p[q] = f32x2{fast_exp2(t[nt][q].x), fast_exp2(t[nt][q].y)};
      bp[nt][2 * q] = static_cast<__bf16>(p[q].x);
      bp[nt][2 * q + 1] = static_cast<__bf16>(p[q].y);
    }
    const f32x2 ps2 = (p[0] + p[1]) + (p[2] + p[3]);  // packed adds
    l[nt] += rows_sum(ps2.x + ps2.y);
  }
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int dt = 0; dt < HD / 16; ++dt)
      o[nt][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(to_bf16x8(c.v[dt]), bp[nt], o[nt][dt], 0, 0, 0);
  reload_v(c);
}

// The (rare) lazy rescale: the running max moves to the chunk max; O and l scale by 2^(m - m_new)
// and the chunk's relative scores t shift by the same amount.
template <int HD, int NT>
__device__ __forceinline__ void full_rescale(const float (&mx)[NT], float (&m)[NT], float (&l)[NT],
                                             f32x4 (&o)[NT][HD / 16], f32x2 (&t)[NT][4]) {
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const bool first = m[nt] == -INFINITY;
    const float m_new = first ? mx[nt] : fmaxf(m[nt], mx[nt]);
    const float alpha = first ? 0.f : fast_exp2(m[nt] - m_new);
    l[nt] *= alpha;
#pragma unroll
    for (int dt = 0; dt < HD / 16; ++dt) o[nt][dt] *= alpha;
    const float shift = m_new - (first ? 0.f : m[nt]);  // t was relative to m_eff (full_scores)
    const f32x2 sh = {shift, shift};
#pragma unroll
    for (int q = 0; q < 4; ++q) t[nt][q] -= sh;
    m[nt] = m_new;
  }
}

template <int HD>
__device__ __forceinline__ void load_q(bf16x8 (&bq)[HD / 32], const bf16_t* row, bool ok, int lane) {
  const int h = lane >> 4;
#pragma unroll
  for (int kk = 0; kk < HD / 32; ++kk) {
    u16x8 v = *reinterpret_cast<const u16x8*>(row + kk * 32 + h * 8);
    if (!ok) v = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
    bq[kk] = __builtin_bit_cast(bf16x8, v);
  }
}

struct AllVisible {
  __device__ bool operator()(int) const { return true; }
};

struct Causal {
  int pos;
  __device__ bool operator()(int t) const { return t <= pos; }
};

// ------------------------------------------------------------------ decode
// Work item = (sequence b, CPW*128-token split, kv head): the 4 waves of a
// workgroup take CPW consecutive 32-token chunks each (all CPW x 16 16-B loads
// issued before the first MFMA), and the G = n_q / n_kv query heads of the kv head
// share every K/V byte (GQA packing).  Items are enumerated from the LIVE
// context lengths -- a prefix sum over ceil(ctx_b / split) computed by every
// workgroup into LDS -- and a fixed grid strides over them.  A grid sized from
// the block-table width instead (graph-safe, but ctx << max_model_len) spent
// most of its workgroups reading seq_lens only to exit: 78 % of the launch at
// B = 160, ctx 1700, max_model_len 8192.
constexpr int DEC_MAX_B = 2048;
constexpr int DEC_MAX_SHARED_SPLITS = 16;   // slots of the shared-prefix pass (bcg_decode_max_splits)

//
// Shared-prefix (cascade) form: rows whose leading blocks are the SAME physical blocks
// (prefix cache: an agent's system prompt, identical in every game) get kv_begin[b] =
// the shared token count and split_base[b] = the shared pass's split count.
// decode_shared_kernel computes their attention over the shared blocks once per group --
// every member's query heads packed into MFMA columns, each shared K/V byte read once per
// 64 columns instead of once per row -- into slots 0 .. split_base-1; this kernel covers
// [kv_begin, ctx) into the slots after them; the combine merges all slots.
// kv_begin == nullptr: no cascade (every row from token 0).

// The projected rows of a step and what its rotary embedding needs (decode_pair_kernel).
struct FusedArgs {
  const bf16_t* qkv;        // [B, n_q + 2 n_kv, HD]
  const int* positions;     // [B]
  const int* slots;         // [B]
  const bf16_t* q_norm;     // [HD] or null
  const bf16_t* k_norm;
  const float* cos_sin;     // [positions, HD]: cos, sin
  float eps;
};

// One head as a row of an operand fragment: lane group h holds dims 32 kk + 8 h .. + 7, and with them both sides of its rotation
// pairs (d, d + HD / 2): normalised, rotated and rounded as qk_norm_rope_kv_vec_kernel does.
template <int HD>
__device__ __forceinline__ void rope_fragments(bf16x8 (&out)[HD / 32], const u16x8 (&raw)[HD / 32], const u16x8 (&norm)[HD / 32],
                                               bool normed, const f32x4 (&cs)[HD / 64][2], const f32x4 (&sn)[HD / 64][2], float eps, int h) {
  constexpr int KK = HD / 32;
  float x[KK][8];
#pragma unroll
  for (int kk = 0; kk < KK; ++kk)
#pragma unroll
    for (int j = 0; j < 8; ++j) x[kk][j] = bf2f(raw[kk][j]);
  if (normed) {
    float ss = 0.f;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
#pragma unroll
      for (int j = 0; j < 8; ++j) ss += x[kk][j] * x[kk][j];
    ss = rows_sum(ss);
    const float inv = rsqrtf(ss / HD + eps);
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
#pragma unroll
      for (int j = 0; j < 8; ++j) x[kk][j] *= inv * bf2f(norm[kk][j]);
  }
#pragma unroll
  for (int kk = 0; kk < KK / 2; ++kk) {
    u16x8 lo, hi;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float c = cs[kk][j >> 2][j & 3], sv = sn[kk][j >> 2][j & 3], x1 = x[kk][j], x2 = x[kk + KK / 2][j];
      lo[j] = f2bf(x1 * c - x2 * sv);
      hi[j] = f2bf(x2 * c + x1 * sv);
    }
    out[kk] = __builtin_bit_cast(bf16x8, lo);
    out[kk + KK / 2] = __builtin_bit_cast(bf16x8, hi);
  }
}

template <int HD>
__device__ __forceinline__ void load_head(u16x8 (&raw)[HD / 32], const bf16_t* row, int h) {
#pragma unroll
  for (int kk = 0; kk < HD / 32; ++kk) raw[kk] = *reinterpret_cast<const u16x8*>(row + kk * 32 + h * 8);
}
// ------------------------------------------------------- decode, streamed
// What the kernel below does when its items are more than one round of workgroups: every wave takes an even share of ALL chunks of the batch, pairs
// (row, kv head) in order, their 32-token chunks in order, cut into as many ranges as there are waves.  A wave's K/V comes by LDS-DMA into 16
// KB of its own: K of the next chunk is fetched when this one's is in registers, V likewise, across pairs, so no fetch waits
// for a pair's table, queries or merge and no wave for another.  What bounds the items (4.6 TB/s at 448 rows of 1050 tokens, heads of 128): between two
// of them the chain of table, loads and merge leaves the memory idle, and the registers hold one item's loads.  A page of K or V is 4 KB
// in one piece, and a pair is cut where a range ends, not every 256 tokens: fewer parts to store and merge.
// 448 rows of 8 kv heads, us for items -> this: 60 tokens 51 -> 44, 250 121 -> 114, 1050 418 -> 370 to 380 (5.2 TB/s, merge and all), 160 rows of 2500
// 340 -> 303, 64 rows of 1050 67 -> 62.  Two chunks ahead with one workgroup a CU (32 KB a wave) is level.
constexpr int STREAM_G = 8;           // query heads of a kv head
constexpr int STREAM_RING = 16384;    // bytes of a wave's chunk: K, then V
constexpr int STREAM_Q = STREAM_G * 256;
constexpr int STREAM_LDS = 4 * (STREAM_RING + 2 * STREAM_Q);   // two workgroups a CU

// The merge learns how many parts a pair is cut into from the partials it reads anyway: whoever has the last part writes PARTS_END as the m of the
// slot behind it.  (A table of the cut, or counts beside the partials, cost it another latency: 0.2 us, 2 to 5 % of a step of short contexts.)
constexpr uint32_t PARTS_END = 0x7fc0e4d1u;   // a NaN that no product of bf16 values makes (their payloads end in 16 zeros)
__device__ __forceinline__ void end_parts(float* m) { *reinterpret_cast<uint32_t*>(m) = PARTS_END; }

// The wave that chunk c of the batch falls to, of `waves` that share `total` chunks: wave w has those from w total / waves on
__device__ __forceinline__ int stream_wave(int c, int total, int waves) {
  return static_cast<int>(((static_cast<uint64_t>(c) + 1) * waves - 1) / total);
}

__device__ __forceinline__ void decode_stream(
    unsigned char* smem, const bf16_t* q, const KVGeom& g, const int* block_tables, int max_blocks, const int* seq_lens, int B, int n_q,
    float scale_log2, float* part_o, float* part_ml, int max_splits, const int* kv_begin, const int* split_base) {
  asm("" : "+s"(B));   // the items' row predicates are not kept for the loop below: 8 pairs of scalars that went through vector lanes, 0.2 us of their path
  constexpr int HD = 128;
  static_assert(sizeof(int) * (DEC_MAX_B + 1 + 8) <= STREAM_LDS, "the row table lies where the ring is later");
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, h = lane >> 4;
  const int G = n_q / g.n_kv, slots = max(2, max_splits - (kv_begin ? DEC_MAX_SHARED_SPLITS : 0));
  auto own_chunks = [&](int b) { return (max(0, seq_lens[b] - (kv_begin ? kv_begin[b] : 0)) + CHUNK - 1) / CHUNK; };

  // ---- chunks of the rows before each row, and this wave's range ----
  int b, n, kvh, c, left;          // row, its chunks a head; head; chunk in the pair; chunks of the range
  int part;                        // which part of its pair the wave's first one is
  int gw;                          // its range
  {
    int* pre = reinterpret_cast<int*>(smem);
    int* wsum = pre + DEC_MAX_B + 1;
    constexpr int PER_MAX = DEC_MAX_B / 256;
    const int rows = (B + 255) / 256;
    int cnt[PER_MAX], sum = 0, longest = 0;
#pragma unroll
    for (int j = 0; j < PER_MAX; ++j) {
      const int i = tid * rows + j;
      cnt[j] = j < rows && i < B ? own_chunks(i) : 0;
      sum += cnt[j];
      longest = max(longest, cnt[j]);
    }
    longest = wave_max(longest);
    int incl = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(incl, o, WAVE);
      if (lane >= o) incl += v;
    }
    if (lane == 63) wsum[w] = incl, wsum[4 + w] = longest;
    __syncthreads();
    for (int ww = 0; ww < 4; ++ww) longest = max(longest, wsum[4 + ww]);
    int base = incl - sum;
    for (int ww = 0; ww < w; ++ww) base += wsum[ww];
#pragma unroll
    for (int j = 0; j < PER_MAX; ++j) {
      const int i = tid * rows + j;
      if (j < rows && i < B) pre[i] = base;
      base += cnt[j];
    }
    if (tid == 255) pre[B] = base;
    __syncthreads();
    const int total = pre[B] * g.n_kv;
    // ranges are so long that a pair of n chunks, cut into (n - 2) / shortest + 2 parts at most, has a slot for each
    const int shortest = max(1, (longest + slots - 2) / (slots - 1));
    const int waves = max(1, min(static_cast<int>(gridDim.x) * 4, total / shortest));
    // (neighbouring ranges to the waves of a workgroup: their pages lie side by side; fewer ranges than waves: spread evenly)
    const int at = static_cast<int>(blockIdx.x) * 4 + w, all = gridDim.x * 4;
    gw = at * waves / all;
    const int start = static_cast<int>(static_cast<uint64_t>(gw) * total / waves);
    left = at == 0 || (at - 1) * waves / all != gw ? static_cast<int>((static_cast<uint64_t>(gw) + 1) * total / waves) - start : 0;
    int lo = 0, hi = B - 1;   // the last row that starts at or before `start`
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (pre[mid] * g.n_kv <= start) lo = mid; else hi = mid - 1;
    }
    b = lo;
    n = pre[lo + 1] - pre[lo];
    const int in = start - pre[lo] * g.n_kv;
    kvh = n > 0 ? in / n : 0;
    c = in - kvh * n;
    part = left > 0 ? gw - stream_wave(start - c, total, waves) : 0;
    b = __builtin_amdgcn_readfirstlane(b), n = __builtin_amdgcn_readfirstlane(n), kvh = __builtin_amdgcn_readfirstlane(kvh);
    c = __builtin_amdgcn_readfirstlane(c), part = __builtin_amdgcn_readfirstlane(part);
    left = __builtin_amdgcn_readfirstlane(left);
    __syncthreads();          // the table is read: the ring may be filled
  }
  if (left <= 0) return;      // (no barrier below)

  // ---- fetches.  K piece i of page e: rows 4 i + lane / 16, their 16-byte chunk x at place x ^ f with f = 8 e + 4 (i / 2) + lane / 16, so that the
  // 16 rows of a fragment read hit 16 places; V^T piece i: rows 32 i + lane / 2, halves swapped where bit 3 of the row is set.
  uint32_t off_k[2][4], off_v[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int e = 0; e < 2; ++e) off_k[e][i] = (4 * i + h) * 256 + ((r ^ (8 * e + 4 * (i >> 1) + h)) << 4);
    off_v[i] = i * 1024 + (lane >> 1) * 32 + (((lane ^ (lane >> 4)) & 1) << 4);
  }
  const uint32_t lds = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem));
  const uint32_t ring = lds + w * STREAM_RING, qring = lds + 4 * STREAM_RING + w * 2 * STREAM_Q;
  auto dma = [&](uint32_t off, const unsigned char* base, uint32_t to) {   // (s_nop: the wait state of an LDS load behind a scalar write of m0)
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "s"(to) : "memory", "m0");
  };
  const unsigned char* kc = reinterpret_cast<const unsigned char*>(g.k);
  const unsigned char* vc = reinterpret_cast<const unsigned char*>(g.v);
  auto page = [&](int blk, int head) {
    return ((static_cast<size_t>(g.layer) * g.num_blocks + blk) * g.n_kv + head) * (BS * HD * 2);
  };
  // (constant address space: scalar loads.  Behind the asm of the fetches hipcc takes vector loads for them, whose wait drains the ring.)
  typedef const __attribute__((address_space(4))) int* Ints;
  auto ints = [](const int* p) { return reinterpret_cast<Ints>(reinterpret_cast<uintptr_t>(p)); };
  const Ints lens = ints(seq_lens), begins = ints(kv_begin), tables = ints(block_tables), bases = ints(split_base);
  struct Row {
    Ints table;   // from the row's first own block on
    int ctx, begin, last, n;   // tokens, first own token, last entry of `table`, chunks a head
  };
  auto row = [&](int i) {
    Row x;
    x.begin = kv_begin ? begins[i] : 0;
    x.ctx = lens[i];
    x.table = tables + static_cast<size_t>(i) * max_blocks + x.begin / BS;
    x.last = (x.ctx - 1) / BS - x.begin / BS;
    x.n = (max(0, x.ctx - x.begin) + CHUNK - 1) / CHUNK;
    return x;
  };
  struct Cursor {
    Row x;
    int b, kvh, c, pair;
  };
  auto advance = [&](Cursor& k) {
    if (++k.c < k.x.n) return;
    k.c = 0;
    k.pair ^= 1;
    if (++k.kvh < g.n_kv) return;
    k.kvh = 0;
    do {   // (only called with chunks left: a row that has some follows)
      ++k.b;
      k.x = row(k.b);
    } while (k.x.n == 0 && k.b < B - 1);
  };
  Cursor use = {row(b), b, kvh, c, 0}, get = use;
  int togo = left;            // chunks not yet fetched
  int blk0 = 0, blk1 = 0;     // pages of the chunk that is fetched next
  auto look = [&]() {
    blk0 = get.x.table[2 * get.c];
    blk1 = get.x.table[min(2 * get.c + 1, get.x.last)];
  };
  auto fetch_k = [&](bool fresh) {
    if (get.c == 0 || fresh) {   // the pair's queries (rows past the heads repeat the last and are not used)
      const unsigned char* qs = reinterpret_cast<const unsigned char*>(q + (static_cast<size_t>(get.b) * n_q + get.kvh * G) * HD);
      dma(min(h, G - 1) * 256 + r * 16, qs, qring + get.pair * STREAM_Q);
      if (G > 4) dma(min(4 + h, G - 1) * 256 + r * 16, qs, qring + get.pair * STREAM_Q + 1024);
    }
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int i = 0; i < 4; ++i) dma(off_k[e][i], kc + page(e ? blk1 : blk0, get.kvh), ring + e * 4096 + i * 1024);
  };
  auto fetch_v = [&]() {
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int i = 0; i < 4; ++i) dma(off_v[i], vc + page(e ? blk1 : blk0, get.kvh), ring + 8192 + e * 4096 + i * 1024);
    --togo;
    if (togo > 0) {
      advance(get);
      look();
    }
  };

  look();
  fetch_k(true);
  fetch_v();

  const unsigned char* rk = smem + w * STREAM_RING + (8 * (r >> 2) + (r & 3)) * 256;
  const unsigned char* rv = smem + w * STREAM_RING + 8192 + (h >> 1) * 4096 + r * 32 + (((h ^ (r >> 3)) & 1) << 4);
  bf16x8 bq[HD / 32];
  float m = -INFINITY, l = 0.f;
  f32x4 o[HD / 16];
  bool fresh = true;
  for (; left > 0; --left) {
    Chunk<HD> x;
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory");   // all but this chunk's V (stores among them only make the wait longer)
    if (fresh) {
      const unsigned char* rq = smem + 4 * STREAM_RING + (w * 2 + use.pair) * STREAM_Q + (r & 7) * 256 + h * 16;
#pragma unroll
      for (int kk = 0; kk < HD / 32; ++kk) {
        bf16x8 v = *reinterpret_cast<const bf16x8*>(rq + kk * 64);
        bq[kk] = r < G ? v : bf16x8{};
      }
      m = -INFINITY, l = 0.f;
#pragma unroll
      for (int dt = 0; dt < HD / 16; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
      fresh = false;
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int kk = 0; kk < HD / 32; ++kk) x.k[u][kk] = *reinterpret_cast<const bf16x8*>(rk + u * 1024 + (((kk * 4 + h) ^ r) << 4));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (togo > 0) {
      fetch_k(false);
      asm volatile("s_waitcnt vmcnt(8)" ::: "memory");   // all but the next chunk's K
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
#pragma unroll
    for (int dt = 0; dt < HD / 16; ++dt) x.v[dt] = *reinterpret_cast<const bf16x8*>(rv + dt * 512);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (togo > 0) fetch_v();
    const int tj = use.x.begin + use.c * CHUNK;
    if (tj + CHUNK <= use.x.ctx)  // wave-uniform: a full chunk needs no tail masking
      compute_chunk<HD, AllVisible, false>(x, bq, tj, use.x.ctx, AllVisible{}, scale_log2, m, l, o, lane);
    else
      compute_chunk<HD, AllVisible, true>(x, bq, tj, use.x.ctx, AllVisible{}, scale_log2, m, l, o, lane);
    if (left == 1 || use.c + 1 == use.x.n) {   // the pair or the range ends
      if (r < G) {
        const int slot = (split_base ? bases[use.b] : 0) + part;
        const size_t at = (static_cast<size_t>(use.b) * n_q + use.kvh * G + r) * max_splits + slot;
#pragma unroll
        for (int dt = 0; dt < HD / 16; ++dt) *reinterpret_cast<f32x4*>(part_o + at * HD + dt * 16 + 4 * h) = o[dt];
        if (h == 0) *reinterpret_cast<float2*>(part_ml + at * 2) = float2{m, l};
        if (h == 0 && use.c + 1 == use.x.n && slot + 1 < max_splits) end_parts(part_ml + (at + 1) * 2);
      }
      part = 0;
      fresh = true;
    }
    if (left > 1) advance(use);
  }
}

template <int HD>
struct ItemShared {
  int pre[DEC_MAX_B + 1];
  int wsum[DEC_WAVES];
  float ml[DEC_WAVES][2][16];
  float o[DEC_WAVES][HD][16 + 1];
};
// STREAM: a step of more items than workgroups is streamed (heads of 128 in bf16)
template <int HD, bool F8 = false, int CPW = 1, bool STREAM = false>
__global__ __launch_bounds__(256, (STREAM ? 2 : 1)) void decode_attn_kernel(
    const bf16_t* __restrict__ q, KVGeom g, const int* __restrict__ block_tables, int max_blocks,
    const int* __restrict__ seq_lens, int B, int n_q, float scale_log2, float* __restrict__ part_o,
    float* __restrict__ part_ml, int max_splits, const int* __restrict__ kv_begin,
    const int* __restrict__ split_base) {
  static_assert(!STREAM || (HD == 128 && !F8), "streamed: decode_stream");
  // CPW chunks per wave: an item covers DEC_WAVES * CPW * 32 tokens; every chunk's loads of
  // a wave are issued before its first MFMA (CPW x 16 loads in flight per wave), and the
  // split partials / merge traffic shrink by CPW
  constexpr int DEC_SPLIT = DEC_WAVES * CHUNK * CPW;
  constexpr int LDS = STREAM ? std::max<int>(STREAM_LDS, sizeof(ItemShared<HD>)) : sizeof(ItemShared<HD>);
  __shared__ __attribute__((aligned(1024))) unsigned char smem[LDS];
  ItemShared<HD>& shared = *reinterpret_cast<ItemShared<HD>*>(smem);
  auto &s_pre = shared.pre;
  auto &s_wsum = shared.wsum;
  auto &s_ml = shared.ml;
  auto &s_o = shared.o;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int r = lane & 15, h = lane >> 4;
  const int G = n_q / g.n_kv;

  // ---- item enumeration: s_pre[b] = sum_{b' < b} ceil(ctx_b' / 128)
  {
    constexpr int PER_MAX = DEC_MAX_B / 256;
    const int per = (B + 255) / 256;  // <= PER_MAX
    int cnt[PER_MAX], sum = 0;
#pragma unroll
    for (int j = 0; j < PER_MAX; ++j) {
      const int i = tid * per + j;
      const int own = (j < per && i < B) ? max(0, seq_lens[i] - (kv_begin ? kv_begin[i] : 0)) : 0;
      cnt[j] = (own + DEC_SPLIT - 1) / DEC_SPLIT;
      sum += cnt[j];
    }
    int incl = sum;  // inclusive wave scan
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(incl, o, WAVE);
      if (lane >= o) incl += v;
    }
    if (lane == 63) s_wsum[w] = incl;
    __syncthreads();
    int base = incl - sum;
    for (int ww = 0; ww < w; ++ww) base += s_wsum[ww];
#pragma unroll
    for (int j = 0; j < PER_MAX; ++j) {
      const int i = tid * per + j;
      if (j < per && i < B) s_pre[i] = base;
      base += cnt[j];
    }
    if (tid == 255) s_pre[B] = base;
    __syncthreads();
  }
  const int n_items = s_pre[B] * g.n_kv;
  if constexpr (STREAM) {
    // One round of items is shorter (16 rows, 2 kv heads, 250 to 1700 tokens: 11.5 to 14 us, streamed 15 to 18), more than one are not (from 590
    // items on 0.84 to 0.99 of the time, 480 still 1.1): only the device knows the contexts.
    if (n_items > static_cast<int>(gridDim.x)) {
      __syncthreads();
      decode_stream(smem, q, g, block_tables, max_blocks, seq_lens, B, n_q, scale_log2, part_o, part_ml, max_splits, kv_begin, split_base);
      return;
    }
  }

  for (int item = blockIdx.x; item < n_items; item += gridDim.x) {
    const int pos = item / g.n_kv, kvh = item - pos * g.n_kv;
    int lo = 0, hi = B - 1;  // last b with s_pre[b] <= pos (binary search, wave-uniform)
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (s_pre[mid] <= pos) lo = mid; else hi = mid - 1;
    }
    const int b = lo, split = pos - s_pre[b];
    const int ctx = seq_lens[b];
    const int start = (kv_begin ? kv_begin[b] : 0) + split * DEC_SPLIT;
    const int slot = (split_base ? split_base[b] : 0) + split;  // after the shared-pass slots
    const int* table = block_tables + static_cast<size_t>(b) * max_blocks;

    bf16x8 bq[HD / 32];
    load_q<HD>(bq, q + (static_cast<size_t>(b) * n_q + kvh * G + (r < G ? r : 0)) * HD, r < G, lane);
    float m = -INFINITY, l = 0.f;
    f32x4 o[HD / 16];
#pragma unroll
    for (int dt = 0; dt < HD / 16; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int t0 = start + w * CHUNK * CPW;
    const int last_blk = (ctx - 1) / BS;
    Chunk<HD, F8> c[CPW];
#pragma unroll
    for (int j = 0; j < CPW; ++j) {
      const int tj = t0 + j * CHUNK;
      if (tj < ctx)  // wave-uniform
        load_chunk<HD, F8>(c[j], g, table[tj / BS], table[min(tj / BS + 1, last_blk)], kvh, lane);
    }
#pragma unroll
    for (int j = 0; j < CPW; ++j) {
      const int tj = t0 + j * CHUNK;
      if (tj >= ctx) break;  // wave-uniform
      if (tj + CHUNK <= ctx)  // wave-uniform: a full chunk needs no tail masking
        compute_chunk<HD, AllVisible, false, F8>(c[j], bq, tj, ctx, AllVisible{}, scale_log2, m, l, o, lane);
      else
        compute_chunk<HD, AllVisible, true, F8>(c[j], bq, tj, ctx, AllVisible{}, scale_log2, m, l, o, lane);
    }

    // combine the 4 waves through LDS
    if (h == 0) {
      s_ml[w][0][r] = m;
      s_ml[w][1][r] = l;
    }
#pragma unroll
    for (int dt = 0; dt < HD / 16; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) s_o[w][dt * 16 + 4 * h + i][r] = o[dt][i];
    __syncthreads();
    for (int idx = tid; idx < G * HD; idx += blockDim.x) {
      const int qi = idx / HD, d = idx % HD;
      float mm = -INFINITY;
#pragma unroll
      for (int ww = 0; ww < DEC_WAVES; ++ww) mm = fmaxf(mm, s_ml[ww][0][qi]);
      float ll = 0.f, oo = 0.f;
#pragma unroll
      for (int ww = 0; ww < DEC_WAVES; ++ww) {
        const float mw = s_ml[ww][0][qi];
        const float f = mw == -INFINITY ? 0.f : exp2f(mw - mm);
        ll += s_ml[ww][1][qi] * f;
        oo += s_o[ww][d][qi] * f;
      }
      const size_t pidx = (static_cast<size_t>(b) * n_q + kvh * G + qi) * max_splits + slot;
      part_o[pidx * HD + d] = oo;
      if (d == 0) {
        part_ml[pidx * 2] = mm;
        part_ml[pidx * 2 + 1] = ll;
        if constexpr (STREAM) {
          if (pos + 1 == s_pre[b + 1] && slot + 1 < max_splits) end_parts(part_ml + (pidx + 1) * 2);
        }
      }
    }
    __syncthreads();  // s_o / s_ml are rewritten by the next item
  }
}

// ------------------------------------------------------- decode, a workgroup per pair
// Rotary embedding, cache write, attention and merge of a (row, kv head) pair in ONE workgroup: its waves take the pair's 32-token chunks in
// turns and meet in LDS once.  Against rotary launch, items and merge launch it saves two launches (2.5 to 3 us each), the parts' way through
// memory and the items' search for their row (scan, table and loads in a chain).  K/V come by LDS-DMA, a KB in one piece (fragments that
// lanes load from the pages themselves are 16 bytes of a row each, 36 B/ns of a CU; this way 100 where the lines are in a cache), each wave's into
// a chunk of its own, fetched again as soon as it is in registers.  The newest token is a chunk of its own, made of the projected row while
// the first fetches are in flight: the cache counts up to the token before it.  What bounds it: up to 256 pairs the 64 KB that a CU has in flight
// against the memory's latency, past that the memory (5.3 to 5.6 TB/s).
// us, rotary + items or stream + merge -> this (spread lengths, heads of 128 / groups of 4 to 6): 10 rows of 1100 tokens, 8 kv heads 22.2 -> 16.6
// (rows in 2 to 4 parts; whole: 21), 20 of 1500 37.5 -> 30.3, 32 of 400 26.9 -> 16, 101 of 1000 96 -> 86, 448 of 1050 390 -> 362, 400 of 60 47 -> 38; heads of 64, 2 kv heads (items
// that rotate by themselves, merge): 4 of 500 10.5 -> 6.1, 512 of 1000 73 -> 55.
// Waves of a workgroup, chunks of a CU the same throughout (128 KB): fewer for many pairs, whose prologues then hide behind other pairs.  Heads of 128, 4 and
// 2 waves: 800 pairs of 1000 tokens 85.7, 88.9, of 60 16.1, 11.9; 1600 of 2000 307, 311, of 60 31, 22.8.  Heads of 64, 8 and 4: 512 pairs of 1000
// 29.4, 30.1, of 60 7.0, 6.5; 1024 of 1000 55.9, 54.8, of 60 12.1, 9.0.  Twice the waves in one workgroup a CU were level and 1 to 3 us slower for short contexts.
template <int HD, int WAVES>
struct Pair {
  static constexpr int PIECES = HD / 32;               // KB of a page of K or of V
  static constexpr int RING = 4 * PIECES * 1024;       // bytes of a wave's chunk: two pages of K, two of V
  static constexpr int QUERIES = 16 * HD * 2;
  static constexpr int LDS = WAVES * RING + QUERIES;
  static_assert((HD * 17 + 64) * 4 <= RING, "the parts of the waves lie where the chunks were");
  static_assert((16 + 64 * 48 + 16) * 4 <= LDS, "and the factors of up to 64 parts of a row");
};

template <int HD, int NW>
__global__ __launch_bounds__(64 * NW, HD == 64 ? 4 : 2) void decode_pair_kernel(
    KVGeom g, const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ seq_lens, int B, int n_q, float scale_log2,
    const PartRule rule, float* __restrict__ part_o, int* __restrict__ counters, bf16_t* __restrict__ out, FusedArgs fa, const int* __restrict__ order) {
  constexpr int KP = Pair<HD, NW>::PIECES, RING = Pair<HD, NW>::RING, PAGE = HD * BS * 2;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[Pair<HD, NW>::LDS];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, h = lane >> 4;
  // (constant address space: scalar loads, whose wait is not one for the fetches)
  typedef const __attribute__((address_space(4))) int* Ints;
  auto ints = [](const int* p) { return reinterpret_cast<Ints>(reinterpret_cast<uintptr_t>(p)); };
  const Place place = place_of(rule, blockIdx.x, B * g.n_kv);
  const int G = n_q / g.n_kv, at_row = place.at / g.n_kv, kvh = place.at - at_row * g.n_kv;
  auto chunks_of = [&](int n) { return (min(max(n, 0), max_blocks * BS) + CHUNK - 1) / CHUNK; };
  auto chunks = [&](int i) { return chunks_of(seq_lens[i]); };
  Share sh{place.own ? order ? ints(order)[at_row] : at_row : -1, 0, 1, 0};
  if (__builtin_expect(rule.extra > 0 && (sh.row < 0 || rule.each == 0 || chunks_of(ints(seq_lens)[sh.row]) > rule.one), 0)) {
    sh = find_share(rule, B, g.n_kv, sh.row, at_row, chunks);
    if (sh.row < 0) return;   // (the whole workgroup)
  }
  const int b = sh.row, part = sh.part, parts = sh.n;
  const Ints table = ints(block_tables) + static_cast<size_t>(b) * max_blocks;
  const int ctx = min(ints(seq_lens)[b], max_blocks * BS), slot = ints(fa.slots)[b];
  const int all = (ctx + CHUNK - 1) / CHUNK, last = max(ctx - 1, 0) / BS;
  const int start = part * all / parts, nchunk = (part + 1) * all / parts;   // the part's chunks
  const int first = start + (w + NW - 2) % NW;   // (the two waves that rotate begin later: theirs are the last chunks of a turn)
  int at0 = table[min(2 * first, last)], at1 = table[min(2 * first + 1, last)];

  // ---- fetches.  A row of K lies in LDS with its 16-byte pieces permuted so that the 16 rows of a fragment read hit 16 places: piece x of fragment row
  // r at place x ^ r (heads of 128: rows of 16 places) or x ^ (r / 2) (heads of 64: rows of 8, neighbours in the other half); V^T: the
  // halves of a row swapped where bit 3 of it is set.
  uint32_t off_k[2][KP], off_v[KP];
#pragma unroll
  for (int i = 0; i < KP; ++i) {
#pragma unroll
    for (int e = 0; e < 2; ++e)
      off_k[e][i] = HD == 128 ? (4 * i + h) * 256 + ((r ^ (8 * e + 4 * (i >> 1) + h)) << 4)
                              : (8 * i + (lane >> 3)) * 128 + (((lane & 7) ^ (4 * e + 2 * i + (h & 1))) << 4);
    off_v[i] = i * 1024 + (lane >> 1) * 32 + (((lane ^ (lane >> 4)) & 1) << 4);
  }
  const uint32_t ring = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem)) + w * RING;
  auto dma = [&](uint32_t off, const unsigned char* base, uint32_t to) {   // (s_nop: the wait state of an LDS load behind a scalar write of m0)
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "s"(to) : "memory", "m0");
  };
  const unsigned char* kc = reinterpret_cast<const unsigned char*>(g.k);
  const unsigned char* vc = reinterpret_cast<const unsigned char*>(g.v);
  auto page = [&](int blk) { return block_base<HD>(g, blk, kvh) * 2; };
  auto fetch_k = [&](int blk0, int blk1) {
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int i = 0; i < KP; ++i) dma(off_k[e][i], kc + page(e ? blk1 : blk0), ring + e * PAGE + i * 1024);
  };
  auto fetch_v = [&](int blk0, int blk1) {
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int i = 0; i < KP; ++i) dma(off_v[i], vc + page(e ? blk1 : blk0), ring + (2 + e) * PAGE + i * 1024);
  };
  auto begin = [&]() {
    if (first < nchunk) {
      fetch_k(at0, at1);   // (a chunk of one page reads it twice)
      fetch_v(at0, at1);
    }
  };
  if (w >= 2) begin();

  // ---- the first wave rotates the queries, the second of the last part the new key, which it stores with the value
  bf16_t* queries = reinterpret_cast<bf16_t*>(smem + NW * RING);   // [16][HD]
  bool own = false;    // (a parked row stores elsewhere than it reads: its newest token is what the cache holds)
  const int newest = max(ctx - 1, 0);
  if (ctx > 0) own = slot == table[newest / BS] * BS + newest % BS;
  const int cached = own ? newest : ctx;
  const bool adds = w == 1 && part == parts - 1;
  Chunk<HD> x;
  if (w == 0 || adds) {
    const bf16_t* heads = fa.qkv + static_cast<size_t>(b) * (n_q + 2 * g.n_kv) * HD;
    const bf16_t* nw = w == 0 ? fa.q_norm : fa.k_norm;
    u16x8 raw[HD / 32], wn[HD / 32] = {};
    f32x4 cs[HD / 64][2], sn[HD / 64][2];
    bf16_t nv[HD / 16];
    load_head<HD>(raw, heads + (w == 0 ? kvh * G + (r < G ? r : 0) : n_q + kvh) * HD, h);
    if (nw != nullptr) load_head<HD>(wn, nw, h);
    if (w == 1) {
#pragma unroll
      for (int dt = 0; dt < HD / 16; ++dt) nv[dt] = heads[(n_q + g.n_kv + kvh) * HD + dt * 16 + r];
    }
    const float* t = fa.cos_sin + static_cast<size_t>(ints(fa.positions)[b]) * HD + 8 * h;
#pragma unroll
    for (int kk = 0; kk < HD / 64; ++kk)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        cs[kk][e] = *reinterpret_cast<const f32x4*>(t + kk * 32 + 4 * e);
        sn[kk][e] = *reinterpret_cast<const f32x4*>(t + HD / 2 + kk * 32 + 4 * e);
      }
    bf16x8 turned[HD / 32];
    rope_fragments<HD>(turned, raw, wn, nw != nullptr, cs, sn, fa.eps, h);
    if (w == 0) {
#pragma unroll
      for (int kk = 0; kk < HD / 32; ++kk)
        *reinterpret_cast<bf16x8*>(queries + r * HD + kk * 32 + h * 8) = r < G ? turned[kk] : bf16x8{};
    } else {
      const size_t base = block_base<HD>(g, slot / BS, kvh);
      bf16_t* kd = const_cast<bf16_t*>(g.k) + base + (slot % BS) * HD + 8 * h;
      bf16_t* vd = const_cast<bf16_t*>(g.v) + base + slot % BS;
      if (r == 0) {
#pragma unroll
        for (int kk = 0; kk < HD / 32; ++kk) *reinterpret_cast<bf16x8*>(kd + kk * 32) = turned[kk];
      }
#pragma unroll
      for (int dt = 0; dt < HD / 16; ++dt)
        if (dt % 4 == h) vd[(dt * 16 + r) * BS] = nv[dt];
      // token 0 of a chunk whose others are masked
#pragma unroll
      for (int kk = 0; kk < HD / 32; ++kk) x.k[0][kk] = r == 0 ? turned[kk] : bf16x8{}, x.k[1][kk] = bf16x8{};
#pragma unroll
      for (int dt = 0; dt < HD / 16; ++dt) {
        u16x8 v = {};
        v[0] = nv[dt];
        x.v[dt] = __builtin_bit_cast(bf16x8, v);
      }
    }
  }
  if (w < 2) begin();
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  bf16x8 bq[HD / 32];
#pragma unroll
  for (int kk = 0; kk < HD / 32; ++kk) bq[kk] = *reinterpret_cast<const bf16x8*>(queries + r * HD + kk * 32 + h * 8);
  float m = -INFINITY, l = 0.f;
  f32x4 o[HD / 16];
#pragma unroll
  for (int dt = 0; dt < HD / 16; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (adds && own) compute_chunk<HD, AllVisible, true>(x, bq, 0, 1, AllVisible{}, scale_log2, m, l, o, lane);

  constexpr int K_ROW = HD * 2;
  const unsigned char* rk = smem + w * RING + (8 * (r >> 2) + (r & 3)) * K_ROW;
  const unsigned char* rv = smem + w * RING + 2 * PAGE + (h >> 1) * PAGE + r * 32 + (((h ^ (r >> 3)) & 1) << 4);
  const int swap = HD == 128 ? r : r >> 1;
  for (int j = first; j < nchunk; j += NW) {
    const int next = j + NW;
    at0 = table[min(2 * next, last)];
    at1 = table[min(2 * next + 1, last)];
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * KP) : "memory");   // all but this chunk's V
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int kk = 0; kk < HD / 32; ++kk) x.k[u][kk] = *reinterpret_cast<const bf16x8*>(rk + u * 4 * K_ROW + (((kk * 4 + h) ^ swap) << 4));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (next < nchunk) {
      fetch_k(at0, at1);
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * KP) : "memory");   // all but the next chunk's K
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
#pragma unroll
    for (int dt = 0; dt < HD / 16; ++dt) x.v[dt] = *reinterpret_cast<const bf16x8*>(rv + dt * 512);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (next < nchunk) fetch_v(at0, at1);
    const int tj = j * CHUNK;
    if (tj + CHUNK <= cached)   // wave-uniform: a full chunk needs no tail masking
      compute_chunk<HD, AllVisible, false>(x, bq, tj, cached, AllVisible{}, scale_log2, m, l, o, lane);
    else if (tj < cached)
      compute_chunk<HD, AllVisible, true>(x, bq, tj, cached, AllVisible{}, scale_log2, m, l, o, lane);
  }

  // ---- the waves' parts meet (every fetch has landed: the last chunk of a wave waits for all of its own)
  __syncthreads();
  float* ml = reinterpret_cast<float*>(smem);             // [NW][2][16]
  float* fac = ml + NW * 32;                              // [NW][16] factors of the waves' parts, [16] of their sum
  float* po = fac + NW * 32;                              // [NW][HD][17]
  if (h == 0) {
    ml[w * 32 + r] = m;
    ml[w * 32 + 16 + r] = l;
  }
#pragma unroll
  for (int dt = 0; dt < HD / 16; ++dt)
#pragma unroll
    for (int i = 0; i < 4; ++i) po[(w * HD + dt * 16 + 4 * h + i) * 17 + r] = o[dt][i];
  __syncthreads();
  // where a part of a cut row lies: [2 extra] slots of [G][HD] outputs, then as many of [G][2] maxima and denominators; the first part behind the others
  auto slot_at = [&](int p) { return p > 0 ? (sh.first + p - 1) * g.n_kv + kvh : rule.extra + sh.first * g.n_kv + kvh; };
  auto slot_o = [&](int p) { return part_o + static_cast<size_t>(slot_at(p)) * G * HD; };
  auto slot_ml = [&](int p) { return part_o + (static_cast<size_t>(2 * rule.extra) * HD + 2 * static_cast<size_t>(slot_at(p))) * G; };
  if (tid < G) {
    float mm = -INFINITY;
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) mm = fmaxf(mm, ml[ww * 32 + tid]);
    float ll = 0.f;
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) {
      const float mw = ml[ww * 32 + tid];
      const float f = mw == -INFINITY ? 0.f : exp2f(mw - mm);
      fac[ww * 16 + tid] = f;
      ll += ml[ww * 32 + 16 + tid] * f;
    }
    fac[NW * 16 + tid] = ll > 0.f ? 1.f / ll : 0.f;
    if (parts > 1) {
      store_through(slot_ml(part) + 2 * tid, mm);
      store_through(slot_ml(part) + 2 * tid + 1, ll);
    }
  }
  __syncthreads();
  bf16_t* heads_out = out + (static_cast<size_t>(b) * n_q + kvh * G) * HD;
  for (int idx = tid; idx < G * HD; idx += 64 * NW) {
    const int qi = idx / HD, d = idx % HD;
    float oo = 0.f;
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) oo += po[(ww * HD + d) * 17 + qi] * fac[ww * 16 + qi];
    if (parts == 1) heads_out[idx] = f2bf(oo * fac[NW * 16 + qi]);
    else store_through(slot_o(part) + idx, oo);
  }
  if (parts == 1) return;

  // ---- the last part of a cut row to arrive adds them up, always in their order
  if (!last_of(counters + sh.first * g.n_kv + kvh, parts, reinterpret_cast<int*>(smem))) return;
  const __amdgpu_buffer_rsrc_t rp = __builtin_amdgcn_make_buffer_rsrc(part_o, 0, 2 * rule.extra * G * HD * 4, 0x00020000);
  f32x4 v[8];
  auto load_eight = [&](int p0, int idx) {   // (past the last part: that one again, which is not added; past the heads: zeros)
#pragma unroll
    for (int j = 0; j < 8; ++j)
      v[j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rp, idx < G * HD ? (slot_at(min(p0 + j, parts - 1)) * G * HD + idx) * 4 : -16, 0, 16 /*sc1*/));
  };
  load_eight(0, 4 * tid);   // (beside the maxima)
  float* pml = reinterpret_cast<float*>(smem) + 16;       // [parts][2][16]
  float* pf = pml + parts * 32;                           // [parts][16], [16] of their sum
  for (int i = tid; i < parts * 32; i += 64 * NW) {
    const int p = i >> 5, qi = i & 15;
    if (qi < G) pml[i] = load_through(slot_ml(p) + 2 * qi + ((i >> 4) & 1));
  }
  __syncthreads();
  if (tid < G) {
    float mm = -INFINITY, ll = 0.f;
    for (int p = 0; p < parts; ++p) mm = fmaxf(mm, pml[p * 32 + tid]);
    for (int p = 0; p < parts; ++p) {
      const float mp = pml[p * 32 + tid], f = mp == -INFINITY ? 0.f : exp2f(mp - mm);
      pf[p * 16 + tid] = f;
      ll += pml[p * 32 + 16 + tid] * f;
    }
    pf[parts * 16 + tid] = ll > 0.f ? 1.f / ll : 0.f;
  }
  __syncthreads();
  for (int idx = 4 * tid; idx < G * HD; idx += 256 * NW) {
    const int qi = idx / HD;
    f32x4 oo = {0.f, 0.f, 0.f, 0.f};
    for (int p0 = 0; p0 < parts; p0 += 8) {
      if (p0 > 0 || idx != 4 * tid) load_eight(p0, idx);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (p0 + j < parts) oo += v[j] * pf[(p0 + j) * 16 + qi];
    }
    u16x4 y;
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = f2bf(oo[e] * pf[parts * 16 + qi]);
    *reinterpret_cast<u16x4*>(heads_out + idx) = y;
  }
}

// Rows by their lengths, longest first (equal ones in their order): where more pairs than the CUs hold at once come in the batch's order, the launch ends
// with whichever long ones came late.  us, order of the batch and this (spread by 30 % to either side, heads of 128, 8 kv heads): 101 rows
// of 1000 tokens 86.8, 83.9; 200 of 500 93.2, 91.1; 448 of 1050 375, 362; 64 of 1000, all resident, 55.8, 54.8.  One launch a step, about 4.6 us.
__global__ __launch_bounds__(256) void decode_order_kernel(const int* __restrict__ seq_lens, int B, int* __restrict__ order) {
  __shared__ int before[4][64];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), row = blockIdx.x * 64 + lane;
  const int own = seq_lens[min(row, B - 1)];
  int n = 0;
#pragma unroll 8
  for (int j = w * B / 4; j < (w + 1) * B / 4; ++j) {
    const int other = seq_lens[j];
    n += other > own || (other == own && j < row);
  }
  before[w][lane] = n;
  __syncthreads();
  if (w == 0 && row < B) order[before[0][lane] + before[1][lane] + before[2][lane] + before[3][lane]] = row;
}

// Split merge: one wave per (row, query head), four per workgroup.  Lane s holds split s's
// (m, l) -- all of them fetched by ONE load instruction, reduced with cross-lane ops --
// then every split's O partial (HD floats, one coalesced load per split, HD / 64 per lane)
// is weighted by its factor, broadcast with v_readlane.  The former one-thread-per-dim
// form walked the splits with dependent broadcast loads twice (35 us per layer at B = 616).
constexpr int COMBINE_WAVES = 4;
// STREAM: the parts of a pair that has any end where the attention says (PARTS_END, items alike), else their number follows from the length.
template <int HD, bool STREAM>
__global__ __launch_bounds__(64 * COMBINE_WAVES) void decode_combine_kernel(
    const float* __restrict__ part_o, const float* __restrict__ part_ml, const int* __restrict__ seq_lens, int n_q,
    int max_splits, int split_tokens, int n_bq, bf16_t* __restrict__ out, const int* __restrict__ kv_begin,
    const int* __restrict__ split_base) {
  constexpr int PER = HD / 64;  // dims per lane
  const int lane = threadIdx.x & 63;
  const int bq = blockIdx.x * COMBINE_WAVES + (threadIdx.x >> 6);
  if (bq >= n_bq) return;  // wave-uniform
  const int b = bq / n_q;
  const float2* ml = reinterpret_cast<const float2*>(part_ml) + static_cast<size_t>(bq) * max_splits + lane;
  float2 mlv{-INFINITY, 0.f};
  if (lane < max_splits) mlv = *ml;   // every slot's, before the number of parts is known: what the loads below say arrives at the same time
  const int own = max(0, seq_lens[b] - (kv_begin ? kv_begin[b] : 0));
  // <= max_splits <= 64 (host check); slots 0 .. split_base[b]-1 hold the shared-prefix partials
  const int base = split_base ? split_base[b] : 0;
  int ns = base + (own + split_tokens - 1) / split_tokens;
  if constexpr (STREAM) {   // (a row without tokens has no parts and no end)
    const unsigned long long ends = __ballot(lane >= base && (lane >= max_splits || __builtin_bit_cast(uint32_t, mlv.x) == PARTS_END));
    ns = own == 0 ? base : ends != 0 ? __ffsll(ends) - 1 : 64;
  }
  if (lane >= ns) mlv = float2{-INFINITY, 0.f};
  float mm = mlv.x;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) mm = fmaxf(mm, __shfl_xor(mm, o, 64));
  const float f = mlv.x == -INFINITY ? 0.f : exp2f(mlv.x - mm);
  float ll = mlv.y * f;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) ll += __shfl_xor(ll, o, 64);
  const float* po = part_o + static_cast<size_t>(bq) * max_splits * HD + lane * PER;
  float acc[PER];
#pragma unroll
  for (int e = 0; e < PER; ++e) acc[e] = 0.f;
  int s = 0;
  for (; s + 4 <= ns; s += 4) {  // four splits' loads in flight before their FMAs
    float v[4][PER];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < PER; ++e) v[j][e] = po[(s + j) * HD + e];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float fj = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, f), s + j));
#pragma unroll
      for (int e = 0; e < PER; ++e) acc[e] += fj * v[j][e];
    }
  }
  for (; s < ns; ++s) {
    const float fj = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, f), s));
#pragma unroll
    for (int e = 0; e < PER; ++e) acc[e] += fj * po[s * HD + e];
  }
  const float inv = ll > 0.f ? 1.f / ll : 0.f;
#pragma unroll
  for (int e = 0; e < PER; ++e) out[static_cast<size_t>(bq) * HD + lane * PER + e] = f2bf(acc[e] * inv);
}

// ------------------------------------------------------- decode, shared prefix
// Work item (one wave) = (group, 64-column block, shared split) for the kv head blockIdx.y.  A group's
// columns are its (member, query head) pairs, c = member * G + head, 16 per MFMA tile and
// SH_NT tiles per wave, so the G = n_q / n_kv heads of up to 64 / G rows share every
// 16-B K/V load (the per-row kernel packs only one row's G heads into the 16 columns).
// grp_desc[grp] = {first member in grp_rows, members, shared blocks, unused}; the shared
// block ids are read from the first member's table row (every member holds the same ids
// there).  The shared tokens are all visible to every member (they precede each member's
// own tokens), so the loop is the prefill kernel's full-visibility block (K/V reloaded in
// place, lazy rescale outside the inner loop) plus one masked half chunk for an odd block
// count.  Splitting the shared tokens into split_tokens pieces (own slots) keeps each wave's
// dependent chunk chain short: one whole-prefix item per wave was latency-bound (a 640-token
// prefix = 20 chained chunk loads) and left most SIMDs idle.  Out: slot `split` of each
// member's (m, l, O) partials.  Every table entry is
// range-checked before use: a bad item is skipped, never dereferenced.
constexpr int SH_NT = 4;
constexpr int SH_WAVES = 4;

template <int HD, bool F8>
__global__ __launch_bounds__(64 * SH_WAVES) void decode_shared_kernel(
    const bf16_t* __restrict__ q, KVGeom g, const int* __restrict__ block_tables, int max_blocks, int B, int n_q,
    float scale_log2, const int* __restrict__ grp_rows, int grp_cap, const int* __restrict__ grp_desc,
    int max_groups, const int* __restrict__ items, const int* __restrict__ n_items_p, int max_items,
    int split_tokens, float* __restrict__ part_o, float* __restrict__ part_ml, int max_splits) {
  constexpr int NT = SH_NT;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, h = lane >> 4;
  const int kvh = blockIdx.y;
  const int G = n_q / g.n_kv;
  const int n_items = min(*n_items_p, max_items);
  for (int it = blockIdx.x * SH_WAVES + w; it < n_items; it += gridDim.x * SH_WAVES) {
    const int grp = items[4 * it], cb = items[4 * it + 1], sp = items[4 * it + 2];
    if (grp < 0 || grp >= max_groups || cb < 0 || sp < 0 || sp >= max_splits) continue;  // wave-uniform
    const int mbeg = grp_desc[4 * grp], nmem = grp_desc[4 * grp + 1], nblk = grp_desc[4 * grp + 2];
    if (mbeg < 0 || nmem <= 0 || mbeg + nmem > grp_cap || nblk <= 0 || nblk > max_blocks) continue;
    const int lead = grp_rows[mbeg];
    if (lead < 0 || lead >= B) continue;
    const int* table = block_tables + static_cast<size_t>(lead) * max_blocks;
    const int S = nblk * BS;
    const int t_lo = sp * split_tokens, t_hi = min(S, t_lo + split_tokens);  // this item's shared tokens
    if (t_lo >= S) continue;
    const int ncol = nmem * G;

    bf16x8 bq[NT][HD / 32];
    int qrow[NT], qhd[NT];  // this lane's column: row and query head (qrow < 0: no column)
    float m[NT], l[NT];
    f32x4 o[NT][HD / 16];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int col = cb * (16 * NT) + nt * 16 + r;
      const int mem = col / G;
      int row = col < ncol ? grp_rows[mbeg + mem] : -1;
      if (row >= B) row = -1;
      const int hq = kvh * G + (col - mem * G);
      load_q<HD>(bq[nt], q + (static_cast<size_t>(row >= 0 ? row : 0) * n_q + (row >= 0 ? hq : 0)) * HD, row >= 0,
                 lane);
      qrow[nt] = row;
      qhd[nt] = hq;
      m[nt] = -INFINITY;
      l[nt] = 0.f;
#pragma unroll
      for (int dt = 0; dt < HD / 16; ++dt) o[nt][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    // absolute chunk indices; split_tokens is a multiple of CHUNK, so only the group's last
    // split can end in a half chunk (odd block count)
    const int nchunk = (t_hi + CHUNK - 1) / CHUNK, n_full = t_hi / CHUNK;
    int c = t_lo / CHUNK;
    Chunk<HD, F8> cur;
    load_chunk<HD, F8>(cur, g, table[2 * c], table[min(2 * c + 1, nblk - 1)], kvh, lane);
    while (c < n_full) {
      f32x2 t[NT][4];
      float mx[NT];
      bool grow = false;
      int b0 = 0, b1 = 0;
      for (; c < n_full; ++c) {
        const int cn = min(c + 1, nchunk - 1);
        b0 = table[2 * cn], b1 = table[min(2 * cn + 1, nblk - 1)];
        grow = full_scores<HD, NT, F8>(cur, bq, scale_log2, m, t, mx,
                                       [&](Chunk<HD, F8>& x) { load_chunk_k<HD, F8>(x, g, b0, b1, kvh, lane); });
        if (grow) break;  // wave-uniform
        full_pv<HD, NT, F8>(cur, t, l, o,
                            [&](Chunk<HD, F8>& x) { load_chunk_v<HD, F8>(x, g, b0, b1, kvh, lane); });
      }
      if (!grow) break;
      full_rescale<HD, NT>(mx, m, l, o, t);
      full_pv<HD, NT, F8>(cur, t, l, o,
                          [&](Chunk<HD, F8>& x) { load_chunk_v<HD, F8>(x, g, b0, b1, kvh, lane); });
      ++c;
    }
    if (c < nchunk) {  // odd block count: the last 16 tokens, masked at S (cur holds that chunk)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        compute_chunk<HD, AllVisible, true, F8>(cur, bq[nt], c * CHUNK, t_hi, AllVisible{}, scale_log2, m[nt],
                                                l[nt], o[nt], lane);
    }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      if (qrow[nt] < 0) continue;
      const size_t pidx = (static_cast<size_t>(qrow[nt]) * n_q + qhd[nt]) * max_splits + sp;
#pragma unroll
      for (int dt = 0; dt < HD / 16; ++dt)
        *reinterpret_cast<f32x4*>(part_o + pidx * HD + dt * 16 + 4 * h) = o[nt][dt];
      if (h == 0) {
        part_ml[pidx * 2] = m[nt];
        part_ml[pidx * 2 + 1] = l[nt];
      }
    }
  }
}

struct Cascade {
  const int* kv_begin;    // [B] shared tokens per row (0: none)
  const int* split_base;  // [B] shared-pass splits of the row (its partial slots 0 .. split_base-1)
  const int* grp_rows;    // [grp_cap] members, grouped
  int grp_cap;
  const int* grp_desc;    // [max_groups, 4]
  int max_groups;
  const int* items;       // [max_items, 4] (group, 64-column block, shared split, -)
  const int* n_items;     // [1] live items (device: graph replays see the current count)
  int max_items;
  int split_tokens;       // shared tokens per item (a multiple of CHUNK)
};

template <int HD, bool F8 = false, int CPW = 1>
void launch_decode(const bf16_t* q, KVGeom g, const int* tables, int max_blocks, const int* seq_lens, int B,
                   int n_q, float sl, float* ws, int max_splits, bf16_t* out, const Cascade& cas,
                   hipStream_t stream) {
  constexpr int DEC_SPLIT = DEC_WAVES * CHUNK * CPW;
  const int shared_slots = cas.kv_begin ? DEC_MAX_SHARED_SPLITS : 0;
  // Streamed from 256 pairs of row and kv head on (8 or 2 kv heads; times over those of the items): 256 pairs 0.99 to 1.01 up to 1050 tokens, 0.92 at 1700,
  // 0.91 at 8000; 320: 0.99, 0.93, 0.93; 512: 0.95 at 250, 0.94, 0.88.  Below them it varies: 1.01 to 1.03 up to 600 tokens (this instance's items),
  // 160 pairs 1.03 to 1.05 at 1700 to 4000 and 0.96 at 8000, 192 and 224 0.91 to 0.97 there, 64 to 128 0.94 to 1.05 at 2500 and 4000.
  // (With one slot a row's range could be cut into more parts than there are slots.)
  const bool streamed = HD == 128 && !F8 && n_q / g.n_kv <= STREAM_G && B * g.n_kv >= 256 && max_splits - shared_slots >= 2;
  if (!streamed) max_splits = std::min(max_splits, (max_blocks * BS + DEC_SPLIT - 1) / DEC_SPLIT + shared_slots);   // no slot to spare
  float* part_o = ws;
  float* part_ml = ws + static_cast<size_t>(B) * n_q * max_splits * HD;
  if (cas.kv_begin != nullptr && cas.max_items > 0) {
    // grid fixed by the item capacity (graph-safe); the live count is read on the device
    const int per_kv = std::max(1, std::min((cas.max_items + SH_WAVES - 1) / SH_WAVES, 128));
    hipLaunchKernelGGL((decode_shared_kernel<HD, F8>), dim3(per_kv, g.n_kv), dim3(64 * SH_WAVES), 0, stream, q, g,
                       tables, max_blocks, B, n_q, sl, cas.grp_rows, cas.grp_cap, cas.grp_desc, cas.max_groups,
                       cas.items, cas.n_items, cas.max_items, cas.split_tokens, part_o, part_ml, max_splits);
  }
  // fixed (graph-safe) grid striding over the live items: one full wave of resident workgroups
  auto run = [&](auto stream_c) {
    constexpr bool STREAM = decltype(stream_c)::value;
    static int resident = 0;
    if (resident == 0) {
      int per_cu = 0, cus = 0, dev = 0;
      hipGetDevice(&dev);
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, decode_attn_kernel<HD, F8, CPW, STREAM>, 256, 0);
      resident = std::max(1, per_cu) * std::max(1, cus);
    }
    const int grid = static_cast<int>(std::min<long>(static_cast<long>(B) * g.n_kv * max_splits, resident));
    hipLaunchKernelGGL((decode_attn_kernel<HD, F8, CPW, STREAM>), dim3(grid), dim3(256), 0, stream, q, g, tables, max_blocks,
                       seq_lens, B, n_q, sl, part_o, part_ml, max_splits, cas.kv_begin, cas.split_base);
  };
  const int n_bq = B * n_q;
  auto merge = [&](auto stream_c) {
    hipLaunchKernelGGL((decode_combine_kernel<HD, decltype(stream_c)::value>), dim3((n_bq + COMBINE_WAVES - 1) / COMBINE_WAVES),
                       dim3(64 * COMBINE_WAVES), 0, stream, part_o, part_ml, seq_lens, n_q, max_splits, DEC_SPLIT, n_bq,
                       out, cas.kv_begin, cas.split_base);
  };
  if constexpr (HD == 128 && !F8) {
    if (streamed) {
      run(std::true_type{});
      merge(std::true_type{});
      return;
    }
  }
  run(std::false_type{});
  merge(std::false_type{});
}

// ----------------------------------------------------------------- prefill
// tiles[i] = {b, q_begin, q_end} (packed row indices); q rows of sequence b occupy
// [q_start[b], q_start[b+1]) and are its last rows (positions ctx-qlen .. ctx-1).
//
// A workgroup = 4 waves over one 64-row tile.  Each wave owns NT column tiles
// of 16 query rows (16*NT rows) of ONE query head and streams the kv head's
// K/V once for all of them: every 16-B K/V load feeds NT times the MFMAs of
// the one-tile (NT = 1) form, which was load-bound (L2 -> CU) at 120-200 TF/s.
// Waves of a block: 4/NT row groups x NT heads; grid = (tiles, ceil(n_q/NT)).
#ifndef PREFILL_LAZY
#define PREFILL_LAZY false  // measured: see PERF.md (lazy spills at NT = 4)
#endif
#ifndef PREFILL_FULL_BLOCK
#define PREFILL_FULL_BLOCK 1  // fully visible chunks through full_scores / full_pv (lazy rescale outside the inner loop, in-place reload)
#endif
#ifndef PREFILL_LDS_BUILD
#define PREFILL_LDS_BUILD 0  // compile the shared K/V ring form (LDSKV) into this library
#endif
#ifndef PREFILL_LDS
#define PREFILL_LDS 0  // with PREFILL_LDS_BUILD: use the ring by default; BCG_PREFILL_LDS=0/1 overrides at run time
#endif
#ifndef PREFILL_XCD_ORDER
#define PREFILL_XCD_ORDER 0  // default grid order (BCG_PREFILL_XCD_ORDER=0/1 overrides at run time)
#endif
#ifndef PREFILL_WPE
#define PREFILL_WPE 0
#endif
#if PREFILL_WPE
#define PREFILL_ATTR __attribute__((amdgpu_waves_per_eu(PREFILL_WPE, PREFILL_WPE)))
#else
#define PREFILL_ATTR
#endif
// LDSKV (bf16 cache, HD = 128, NT = 4): the 4 waves of a workgroup are 4 consecutive query heads
// (at most 2 kv heads when G >= 2); each 32-token chunk of both kv heads' K and V goes global -> LDS
// ONCE per workgroup by LDS-DMA (8 x 1-KiB pieces per wave), 4-slot ring, issued 2 chunks ahead;
// the in-place reloads of the full-visibility loop then read their fragments from LDS
// (XOR-swizzled K rows: conflict-free ds_read_b128) instead of issuing 16 global loads per wave.
// One raw s_barrier per chunk (all waves share the rows, so they run the same chunks).
__device__ __forceinline__ int kswz(int row) { return ((row & 3) | ((row & 8) >> 1)) << 1; }

template <int HD, int NT, bool F8 = false, bool LDSKV = false>
__global__ __launch_bounds__(256) PREFILL_ATTR void prefill_attn_kernel(
    const bf16_t* __restrict__ q, KVGeom g, const int* __restrict__ block_tables, int max_blocks,
    const int* __restrict__ q_start, const int* __restrict__ seq_lens, const int* __restrict__ tiles,
    int n_q, float scale_log2, bf16_t* __restrict__ out, int n_tiles, int xcd_order) {
  constexpr int RG = 4 / NT;   // row groups per 64-row tile
  constexpr int ROWS = 16 * NT;
  // xcd_order: 1-D grid; workgroup id b runs on XCD b % 8 (round-robin dispatch), so the
  // head groups of one tile are given consecutive ids of ONE XCD -- the query heads that share
  // a kv head then read its K/V through that XCD's L2 together -- while each XCD still walks
  // the tiles in the host's deepest-first order (tile = 8 * local index + XCD).
  int tile, hgrp;
  if (xcd_order) {
    const int hg_n = (n_q + NT - 1) / NT, s = blockIdx.x >> 3;
    tile = (s / hg_n) * 8 + (blockIdx.x & 7);
    hgrp = s % hg_n;
    if (tile >= n_tiles) return;  // padding of the grid to whole XCD rounds
  } else {
    tile = blockIdx.x;
    hgrp = blockIdx.y;
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int qh = hgrp * NT + w / RG;
  if (qh >= n_q) return;  // wave-uniform; no block-level barriers in this kernel
  const int b = tiles[3 * tile], q_begin = tiles[3 * tile + 1], q_end = tiles[3 * tile + 2];
  const int r = lane & 15, h = lane >> 4;
  const int row0 = q_begin + ROWS * (w % RG);
  if (row0 >= q_end) return;
  const int ctx = seq_lens[b];
  const int qs = q_start[b], qlen = q_start[b + 1] - qs;
  const int pos0 = ctx - qlen;  // position of row qs
  const int kvh = qh / (n_q / g.n_kv);
  const int* table = block_tables + static_cast<size_t>(b) * max_blocks;

  bf16x8 bq[NT][HD / 32];
  float m[NT], l[NT];
  f32x4 o[NT][HD / 16];
  // query position of this lane's column; per sub-tile: first row's position, exclusive key bound
  int my_pos[NT], sub_first[NT], sub_end[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int my_row = row0 + 16 * nt + r;
    const bool ok = my_row < q_end;
    load_q<HD>(bq[nt], q + (static_cast<size_t>(ok ? my_row : row0) * n_q + qh) * HD, ok, lane);
    my_pos[nt] = pos0 + (my_row - qs);
    sub_first[nt] = pos0 + (row0 + 16 * nt - qs);
    sub_end[nt] = pos0 + (min(row0 + 16 * nt + 15, q_end - 1) - qs) + 1;
    m[nt] = -INFINITY;
    l[nt] = 0.f;
#pragma unroll
    for (int dt = 0; dt < HD / 16; ++dt) o[nt][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const int last_row = min(row0 + ROWS - 1, q_end - 1);
  const int kv_end = pos0 + (last_row - qs) + 1;  // exclusive bound of keys visible to this wave

  // block ids in windows of 64 (one per lane), broadcast with readlane (see decode)
  const int nblk = (kv_end + BS - 1) / BS;
  int win_base = 0;
  int my_blk = lane < nblk ? table[lane] : 0;
  auto block_at = [&](int bi) -> int {
    if (bi >= win_base + 64) {  // wave-uniform: advance the window
      win_base += 64;
      my_blk = win_base + lane < nblk ? table[win_base + lane] : 0;
    }
    return __builtin_amdgcn_readlane(my_blk, bi - win_base);
  };
  // next-chunk loads issued unconditionally (clamped to the last chunk) -- see decode
  const int nchunk = (kv_end + CHUNK - 1) / CHUNK;
  Chunk<HD, F8> cur;
  load_chunk<HD, F8>(cur, g, block_at(0), block_at(min(1, nblk - 1)), kvh, lane);
#if PREFILL_FULL_BLOCK
  // chunks every row of the wave sees in full: one interleaved block for all NT sub-tiles,
  // the next chunk reloaded in place (K after the S^T MFMAs, V after the P.V MFMAs): no
  // second register set for the prefetch
  int c = 0;
  const int n_full = min(sub_first[0] / CHUNK, nchunk);  // chunks every row of the wave sees in full

  // ---- LDSKV: shared K/V ring (see above the kernel) ----
  constexpr int KV_SLOTS = 4, KV_HALF = 8192, KV_HEAD = 2 * KV_HALF, KV_SLOT = 2 * KV_HEAD;
  __shared__ __attribute__((aligned(1024))) unsigned char kv_ring[LDSKV ? KV_SLOTS * KV_SLOT : 16];
  const int kvA = LDSKV ? (hgrp * NT) / (n_q / g.n_kv) : 0;
  const int kvsel = kvh - kvA;                                              // which staged kv head this wave reads
  const int dkv = min(kvA + (w >> 1), (hgrp * NT + NT - 1) / (n_q / g.n_kv));  // kv head this wave stages
  // block ids of the DMA lookahead: scalar loads (lgkmcnt) -- a vector load here would make every
  // wait on it (vmcnt counts in order) drain the DMA pieces in flight ahead of it
  auto block_at2 = [&](int bi) -> int { return table[__builtin_amdgcn_readfirstlane(bi)]; };
  auto issue_chunk = [&](int k) {  // this wave's 8 pieces (K or V of kv head dkv) of chunk k
    if constexpr (LDSKV && !F8) {
      const int bb0 = block_at2(2 * k), bb1 = block_at2(min(2 * k + 1, nblk - 1));
      unsigned char* dst = kv_ring + (k % KV_SLOTS) * KV_SLOT + (w >> 1) * KV_HEAD + (w & 1) * KV_HALF;
      const unsigned char* kc = reinterpret_cast<const unsigned char*>(g.k);
      const unsigned char* vc = reinterpret_cast<const unsigned char*>(g.v);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const size_t base = 2 * block_base<HD>(g, i < 4 ? bb0 : bb1, dkv);
        const unsigned char* src;
        if ((w & 1) == 0) {  // K rows (i & 3) * 4 + lane / 16; the lane's LDS slot p holds chunk p ^ kswz(row)
          const int row = (i & 3) * 4 + (lane >> 4);
          src = kc + base + row * 256 + ((lane & 15) ^ kswz(row)) * 16;
        } else {  // V^T: a plain copy of the block-head's 4 KiB
          src = vc + base + (i & 3) * 1024 + lane * 16;
        }
        __builtin_amdgcn_global_load_lds(src, dst + i * 1024, 16, 0, 0);
      }
    }
  };
  auto lds_k = [&](Chunk<HD, F8>& x, int k) {
    if constexpr (LDSKV && !F8) {
      const unsigned char* base = kv_ring + (k % KV_SLOTS) * KV_SLOT + kvsel * KV_HEAD;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int t = 8 * (r >> 2) + 4 * u + (r & 3), row = t & 15;
#pragma unroll
        for (int kk = 0; kk < HD / 32; ++kk)
          x.k[u][kk] =
              *reinterpret_cast<const bf16x8*>(base + (t >> 4) * 4096 + row * 256 + ((4 * kk + h) ^ kswz(row)) * 16);
      }
    }
  };
  auto lds_v = [&](Chunk<HD, F8>& x, int k) {
    if constexpr (LDSKV && !F8) {
      const unsigned char* base =
          kv_ring + (k % KV_SLOTS) * KV_SLOT + kvsel * KV_HEAD + KV_HALF + (h >> 1) * 4096 + (h & 1) * 16;
#pragma unroll
      for (int dt = 0; dt < HD / 16; ++dt) x.v[dt] = *reinterpret_cast<const bf16x8*>(base + (dt * 16 + r) * 32);
    }
  };
  if constexpr (LDSKV && !F8) {  // chunks 1 and 2 ahead of the loop; chunk k + 3 is issued in iteration k
    if (1 < min(n_full + 1, nchunk)) issue_chunk(1);
    if (2 < min(n_full + 1, nchunk)) issue_chunk(2);
  }
  // LDSKV: chunks 1 .. n_stage-1 go through the ring -- every full chunk's successor, including
  // the first masked chunk, which the masked loop below then starts from
  const int n_stage = min(n_full + 1, nchunk);
  auto ring_k = [&](Chunk<HD, F8>& x) {
    if (c + 1 >= n_stage) return;  // no successor (the wave's last chunk): nothing to reload
    // this wave's pieces of chunk c+1 landed (chunk c+2's 8 may still fly), then every wave's
    if (c + 2 < n_stage) {
      asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    __builtin_amdgcn_s_barrier();  // ... and every wave is past chunk c-1: its slot is free
    asm volatile("" ::: "memory");
    if (c + 3 < n_stage) issue_chunk(c + 3);
    lds_k(x, c + 1);
  };
  auto ring_v = [&](Chunk<HD, F8>& x) {
    if (c + 1 < n_stage) lds_v(x, c + 1);
  };
  if constexpr (LDSKV && !F8) {
    // no VGPR-destination global load in this loop: with one, the compiler's wait before the
    // S^T MFMAs would be a vmcnt(0) that drains the ring every chunk
    while (c < n_full) {
      f32x2 t[NT][4];
      float mx[NT];
      bool grow = false;
      for (; c < n_full; ++c) {
        grow = full_scores<HD, NT, F8>(cur, bq, scale_log2, m, t, mx, ring_k);
        if (grow) break;  // wave-uniform
        full_pv<HD, NT, F8>(cur, t, l, o, ring_v);
      }
      if (!grow) break;
      full_rescale<HD, NT>(mx, m, l, o, t);
      full_pv<HD, NT, F8>(cur, t, l, o, ring_v);
      ++c;
    }
  } else {
    while (c < n_full) {
      f32x2 t[NT][4];
      float mx[NT];
      bool grow = false;
      int b0 = 0, b1 = 0;
      // inner loop: no VALU on O (it stays in the MFMA accumulators); leaves with S live
      // when a column's max moved enough to need the lazy rescale
      for (; c < n_full; ++c) {
        const int cn = min(c + 1, nchunk - 1);
#ifdef PREFILL_ABL_HOT  // timing ablation only (wrong results): every reload re-reads chunk 0's blocks (L2-hot)
        b0 = block_at(0), b1 = block_at(min(1, nblk - 1));
#else
        b0 = block_at(2 * cn), b1 = block_at(min(2 * cn + 1, nblk - 1));
#endif
        grow = full_scores<HD, NT, F8>(cur, bq, scale_log2, m, t, mx,
                                       [&](Chunk<HD, F8>& x) { load_chunk_k<HD, F8>(x, g, b0, b1, kvh, lane); });
        if (grow) break;  // wave-uniform
        full_pv<HD, NT, F8>(cur, t, l, o,
                            [&](Chunk<HD, F8>& x) { load_chunk_v<HD, F8>(x, g, b0, b1, kvh, lane); });
      }
      if (!grow) break;
      full_rescale<HD, NT>(mx, m, l, o, t);
      full_pv<HD, NT, F8>(cur, t, l, o,
                          [&](Chunk<HD, F8>& x) { load_chunk_v<HD, F8>(x, g, b0, b1, kvh, lane); });
      ++c;
    }
  }
  Chunk<HD, F8> nxt;
  for (; c < nchunk; ++c) {
#else
  Chunk<HD, F8> nxt;
  for (int c = 0; c < nchunk; ++c) {
#endif
    const int cn = min(c + 1, nchunk - 1);
    load_chunk<HD, F8>(nxt, g, block_at(2 * cn), block_at(min(2 * cn + 1, nblk - 1)), kvh, lane);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      if (c * CHUNK >= sub_end[nt]) continue;  // wave-uniform: chunk wholly in this sub-tile's causal future
      if ((c + 1) * CHUNK <= sub_first[nt])     // wave-uniform: every key visible to every row
        compute_chunk<HD, Causal, false, F8, PREFILL_LAZY>(cur, bq[nt], c * CHUNK, sub_end[nt], Causal{my_pos[nt]},
                                                           scale_log2, m[nt], l[nt], o[nt], lane);
      else
        compute_chunk<HD, Causal, true, F8, PREFILL_LAZY>(cur, bq[nt], c * CHUNK, sub_end[nt], Causal{my_pos[nt]},
                                                          scale_log2, m[nt], l[nt], o[nt], lane);
    }
    cur = nxt;
  }
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int my_row = row0 + 16 * nt + r;
    if (my_row >= q_end) continue;
    const float inv = l[nt] > 0.f ? 1.f / l[nt] : 0.f;
    bf16_t* orow = out + (static_cast<size_t>(my_row) * n_q + qh) * HD;
    // O^T rows d = 16dt + 4h + i are this lane's column (query my_row)
#pragma unroll
    for (int dt = 0; dt < HD / 16; ++dt) {
      u16x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = f2bf(o[nt][dt][i] * inv);
      *reinterpret_cast<u16x4*>(orow + dt * 16 + 4 * h) = v;
    }
  }
}

template <int HD, bool F8>
void launch_prefill(int n_tiles, int n_q, const bf16_t* q, KVGeom g, const int* tables, int max_blocks,
                    const int* q_start, const int* seq_lens, const int* tiles, float sl, bf16_t* out,
                    hipStream_t stream) {
#ifndef PREFILL_NT
#define PREFILL_NT 4
#endif
  constexpr int NT = PREFILL_NT;  // 1 and 2 measured slower (PERF.md); the LDS-shared forms were 180-200 TF/s
  const int hg_n = (n_q + NT - 1) / NT;
  static const int xcd_order = [] {
    const char* e = std::getenv("BCG_PREFILL_XCD_ORDER");
    return e ? std::atoi(e) : PREFILL_XCD_ORDER;
  }();
  static const int lds_env = [] {
    const char* e = std::getenv("BCG_PREFILL_LDS");
    return e ? std::atoi(e) : PREFILL_LDS;
  }();
  // the shared K/V ring needs whole 4-head workgroups spanning <= 2 kv heads, HD = 128, bf16 KV
  const bool lds = lds_env && HD == 128 && !F8 && NT == 4 && n_q % 4 == 0 && n_q / g.n_kv >= 2;
  const dim3 grid = xcd_order ? dim3(((n_tiles + 7) / 8) * 8 * hg_n) : dim3(n_tiles, hg_n);
#if PREFILL_LDS_BUILD  // the shared-ring form lost its A/B: only variant builds carry it (-DPREFILL_LDS_BUILD=1)
  if (lds) {
    hipLaunchKernelGGL((prefill_attn_kernel<HD, NT, F8, true>), grid, dim3(256), 0, stream, q, g, tables, max_blocks,
                       q_start, seq_lens, tiles, n_q, sl, out, n_tiles, xcd_order);
    return;
  }
#else
  (void)lds;
#endif
  hipLaunchKernelGGL((prefill_attn_kernel<HD, NT, F8, false>), grid, dim3(256), 0, stream, q, g, tables, max_blocks,
                     q_start, seq_lens, tiles, n_q, sl, out, n_tiles, xcd_order);
}

// ------------------------------------------------- prefill, 32x32 MFMA, LDS-staged K/V
// The 16x16 kernel above holds 510 registers (one wave per SIMD), so nothing hides a wave's
// softmax VALU or its reload latency behind another wave's MFMAs.  This form is built for two
// waves per SIMD (<= 256 registers): a workgroup = NW waves x 32 query rows of ONE query head
// (tiles of 32 * NW rows), K/V of 64-token chunks staged ONCE per workgroup in an NS-slot LDS
// ring by LDS-DMA (32 x 1-KiB pieces per chunk, P = 32 / NW per wave), one s_barrier per chunk.
//
// Swapped products on v_mfma_f32_32x32x16_bf16 (A[m = l&31][k = 8(l>>5)+j], B[k][n = l&31],
// C[m = 8(i>>2) + 4(l>>5) + (i&3)][n = l&31]):
//   S^T = K Q^T     A = K rows from LDS, B = Q fragments in registers (8 x bf16x8);
//   O^T += V^T P^T  A = V^T rows from LDS (the V cache is [hd][16 tokens] per block),
//                   B = P^T straight from the S^T accumulators of the same lane.
// Token permutation (per 32-token tile u): S^T row m = 16s + 8a + 4h + b holds token
// 32u + 16s + 8h + 4a + b, so accumulator i of lane half h is token 32u + 16(i>>3) + 8h + (i&7):
// P.V k-step 2u + (i>>3) takes the lane's own 8 consecutive accumulators as its B operand, and
// the matching V^T operand is ONE 16-byte read (8 consecutive tokens of a V^T row).  No
// cross-lane traffic except one permlane32_swap per chunk for the column max.
// LDS images (no bank conflicts for the 16-lane groups of ds_read_b128):
//   K: row t (token of the chunk) at t * 256, its 16-B chunk p stored at slot p ^ (t & 15);
//   V: block s at 16 KiB + s * 4 KiB, row d at d * 32, 16-B half e stored at e ^ ((d >> 3) & 1).
// The source side of each LDS-DMA lane applies the swizzle (LDS destinations are consecutive).
typedef float f32x16 __attribute__((ext_vector_type(16)));
constexpr int PREFILL32_MAX_BLOCKS = 1024;  // block-table width the 32x32 kernel stages in LDS (16k tokens)

// One 64-token chunk of prefill_attn32_kernel for one wave (32 query columns):
//   attn32_scores  S^T = K Q^T, the column max m_new (the online softmax rescales EVERY chunk:
//                  a data-dependent rescale branch made hipcc copy the 64 O accumulators between
//                  register sets on every chunk -- 64 v_mov_b64 against 32 v_pk_mul here),
//                  O and the partial sums scaled by 2^(m - m_new), t = S * scale - m_new;
//   attn32_pv      P = 2^t, partial row sums, O^T += V^T P^T.
// MASKED: rel_pos = (token of accumulator 0) - (this column's position) (causal mask),
// rel_ctx = (token of accumulator 0) - ctx (V of tokens past the context is zeroed).
// A column's first chunk always holds a visible key (token 0), so m is finite after it.
template <bool MASKED>
__device__ __forceinline__ void attn32_scores(const unsigned char* slot, int k_lane, const bf16x8 (&bq)[8],
                                              float scale_log2, int rel_pos, float& m, float& lsum,
                                              f32x16 (&o)[4], float (&t)[32]) {
  f32x16 s0 = f32x16{}, s1 = f32x16{};
  bf16x8 ka[8][2];
#pragma unroll
  for (int kk = 0; kk < 8; ++kk) {
    const unsigned char* p = slot + (k_lane ^ (kk << 5));
    ka[kk][0] = *reinterpret_cast<const bf16x8*>(p);
    ka[kk][1] = *reinterpret_cast<const bf16x8*>(p + 32 * 256);
  }
  __builtin_amdgcn_sched_barrier(0);  // keep the reads ahead (the scheduler sinks them to their uses)
#pragma unroll
  for (int kk = 0; kk < 8; ++kk) {
    s0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[kk][0], bq[kk], s0, 0, 0, 0);
    s1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[kk][1], bq[kk], s1, 0, 0, 0);
  }
  // the maxima below are asm, in front of which hipcc puts no wait states: 12 from a product of 8 passes to a vector read of its result, what it puts in
  // front of its own.  (Without them the maximum was taken over what the registers held before, in places: right but for the last bit, another one
  // each time, as long as the scores of two chunks are alike.)
  asm volatile("s_nop 11" : "+v"(s0), "+v"(s1));
  // accumulator i of tile u is token 32u + 16(i>>3) + 8h + (i&7)
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    t[i] = s0[i];
    t[16 + i] = s1[i];
  }
  if constexpr (MASKED) {
#pragma unroll
    for (int i = 0; i < 32; ++i)
      if (rel_pos + 32 * (i >> 4) + 16 * ((i >> 3) & 1) + (i & 7) > 0) t[i] = -INFINITY;
  }
  float v = t[0];
#pragma unroll
  for (int i = 1; i < 31; i += 2) v = vmax3(v, t[i], t[i + 1]);
  v = vmax(v, t[31]);
  const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = vmax(__uint_as_float(sw[0]), __uint_as_float(sw[1])) * scale_log2;  // column max (log2 units)
  const float m_new = vmax(m, v);   // finite from the column's first chunk on
  const float alpha = fast_exp2(m - m_new);  // m = -inf: 0
  m = m_new;
  lsum *= alpha;
  const f32x2 al = {alpha, alpha};
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int i = 0; i < 16; i += 2) {
      const f32x2 x = f32x2{o[dt][i], o[dt][i + 1]} * al;
      o[dt][i] = x.x;
      o[dt][i + 1] = x.y;
    }
  const f32x2 sc = {scale_log2, scale_log2}, mm = {m_new, m_new};
#pragma unroll
  for (int i = 0; i < 32; i += 2) {  // two scores per v_pk_fma_f32 (masked: -inf stays -inf)
    const f32x2 x = f32x2{t[i], t[i + 1]} * sc - mm;
    t[i] = x.x;
    t[i + 1] = x.y;
  }
}

template <bool MASKED>
__device__ __forceinline__ void attn32_pv(const unsigned char* slot, int v_lane, int rel_ctx, const float (&t)[32],
                                          float& lsum, f32x16 (&o)[4]) {
  // P = 2^t, lane-local partial row sums (packed adds); P^T operands of the four 16-token k-steps
  bf16x8 bp[4];
  f32x2 ps = {0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 32; i += 2) {
    const f32x2 p = {fast_exp2(t[i]), fast_exp2(t[i + 1])};
    ps += p;
    bp[i >> 3][i & 7] = static_cast<__bf16>(p.x);
    bp[i >> 3][(i & 7) + 1] = static_cast<__bf16>(p.y);
  }
  lsum += ps.x + ps.y;
  // O^T += V^T P^T (k-step s = block s of the chunk, this lane half's 8 tokens); each V operand
  // is read one MFMA ahead
  const unsigned char* vb = slot + v_lane;
  u32x4 va = *reinterpret_cast<const u32x4*>(vb);
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    uint32_t keep[4] = {~0u, ~0u, ~0u, ~0u};
    if constexpr (MASKED) {  // stale bytes past the context may be non-finite: zero them
#pragma unroll
      for (int j2 = 0; j2 < 4; ++j2) {
        const int tk = rel_ctx + 16 * s + 2 * j2;  // token - ctx
        keep[j2] = (tk < 0 ? 0x0000ffffu : 0u) | (tk + 1 < 0 ? 0xffff0000u : 0u);
      }
    }
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
      const int nx = 4 * s + dt + 1;
      u32x4 vn = va;
      if (nx < 16) vn = *reinterpret_cast<const u32x4*>(vb + (nx >> 2) * 4096 + (nx & 3) * 1024);
      if constexpr (MASKED) {
#pragma unroll
        for (int j2 = 0; j2 < 4; ++j2) va[j2] &= keep[j2];
      }
      o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, va), bp[s], o[dt], 0, 0, 0);
      va = vn;
    }
  }
}

template <int NW, int NS>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2))) void prefill_attn32_kernel(
    const bf16_t* __restrict__ q, KVGeom g, const int* __restrict__ block_tables, int max_blocks,
    const int* __restrict__ q_start, const int* __restrict__ seq_lens, const int* __restrict__ tiles, int n_q,
    float scale_log2, bf16_t* __restrict__ out, int n_tiles) {
  constexpr int HD = 128, KC = 64;                   // head dim, tokens per chunk
  constexpr int KBYTES = KC * HD * 2, SLOT = 2 * KBYTES;  // K (then V) image of one chunk: 16 KiB each
  constexpr int P = 32 / NW;                         // 1-KiB DMA pieces per wave per chunk
  static_assert(NW == 4 || NW == 8, "4 or 8 waves");
  static_assert(NS >= 2 && NS <= 4, "ring depth");
  __shared__ __attribute__((aligned(1024))) unsigned char ring[NS * SLOT];

  // XCD-grouped order (1-D grid): workgroup id i runs on XCD i % 8, so kv head i % n_kv puts every
  // query head of a kv head on the same XCD(s) (one XCD per kv head at n_kv = 8), the G heads of
  // one tile next to each other: the K/V chunks they all stage come from that XCD's L2 (+5-8 %
  // over a (tile, head) grid, profiles/r6_prefill32)
  const int G = n_q / g.n_kv;
  const int kvh = blockIdx.x % g.n_kv, rest = blockIdx.x / g.n_kv;
  const int tile = rest / G, qh = kvh * G + rest % G;
  if (tile >= n_tiles) return;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 31, h = lane >> 5;
  const int b = tiles[3 * tile], q_begin = tiles[3 * tile + 1], q_end = tiles[3 * tile + 2];
  const int ctx = seq_lens[b];
  const int pos0 = ctx - (q_start[b + 1] - q_start[b]) - q_start[b];  // position of packed row r = pos0 + r
  const int* table = block_tables + static_cast<size_t>(b) * max_blocks;
  const int nblk = (ctx + BS - 1) / BS;
  const int wg_last = min(q_begin + 32 * NW, q_end) - 1;
  const int nchunk = (pos0 + wg_last + KC) / KC;      // chunks the workgroup stages (uniform)
  const int row0 = q_begin + 32 * w;
  const bool active = row0 < q_end;                   // wave-uniform
  const int w_last = min(row0 + 31, q_end - 1);
  const int w_chunks = active ? (pos0 + w_last + KC) / KC : 0;          // chunks this wave computes
  const int n_full = active ? min((pos0 + row0 + 1) / KC, w_chunks) : 0;  // ... seen in full by all its rows
  // this lane's query column; columns past q_end compute as the tile's last row (never stored)
  const int my_row = min(row0 + col, q_end - 1);
  const int pos_q = pos0 + my_row;

  // ---- LDS-DMA issue of chunk c into slot c % NS (this wave's P pieces) ----
  // The sequence's block ids are staged in LDS once: a scalar load of a table entry per piece
  // (each followed by its lgkmcnt wait) serialised ~8 round trips into every chunk.
  __shared__ int blk_ids[PREFILL32_MAX_BLOCKS];
  for (int i = threadIdx.x; i < 4 * nchunk; i += 64 * NW) blk_ids[i] = table[min(i, nblk - 1)];
  const unsigned char* kc = reinterpret_cast<const unsigned char*>(g.k);
  const unsigned char* vc = reinterpret_cast<const unsigned char*>(g.v);
  const size_t head_base = static_cast<size_t>(g.layer) * g.num_blocks;
  // lane parts of the source offsets (K piece rows 4 (i & 3) + lane / 16 of a block, its 16-B
  // chunk (lane & 15) ^ row; V^T piece rows d = 32 (i & 3) + lane / 2, half (lane & 1) ^ bit 3 of d)
  const int lane_kx = (lane & 15) ^ (lane >> 4), lane_k = (lane >> 4) * 256;
  const int lane_v = (lane >> 1) * 32 + (((lane ^ (lane >> 4)) & 1) << 4);
  auto issue = [&](int c) __attribute__((always_inline)) {
    unsigned char* slot = ring + (c % NS) * SLOT;
    int blk[P];
#pragma unroll
    for (int pi = 0; pi < P; ++pi) blk[pi] = blk_ids[4 * c + (((w * P + pi) & 15) >> 2)];
#pragma unroll
    for (int pi = 0; pi < P; ++pi) {
      const int i = w * P + pi;  // piece 0..31, wave-uniform
      const int r4 = i & 3;
      const size_t base = ((head_base + __builtin_amdgcn_readfirstlane(blk[pi])) * g.n_kv + kvh) * (BS * HD * 2);
      // K rows 4i .. 4i+3 of the chunk, or V^T rows 32 (i & 3) .. + 31 of block (i & 15) / 4.
      // The DMA as inline asm (M0 = the piece's LDS address): hipcc tracks the builtin's LDS write
      // and put a vmcnt(0) before the next ds_read of the ring -- every chunk then waited for its
      // successor's pieces to land (+4-6 % without).  The ring's own counted wait + barrier in
      // sync() orders the reads.
      const unsigned char* src = i < 16 ? kc + base + (r4 * 1024 + lane_k + ((lane_kx ^ (4 * r4)) << 4))
                                        : vc + base + (r4 * 1024 + lane_v);
      const uint32_t m0v = __builtin_amdgcn_readfirstlane(
          static_cast<uint32_t>(reinterpret_cast<uintptr_t>(slot + (i < 16 ? i * 1024 : KBYTES + (i - 16) * 1024))));
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(src), "s"(m0v) : "memory", "m0");
    }
  };

  // Q^T operands: lane (col, h) holds dims 16 kk + 8 h .. + 7 of its row
  bf16x8 bq[HD / 16];
  {
    const bf16_t* qrow = q + (static_cast<size_t>(my_row) * n_q + qh) * HD + 8 * h;
    u32x4 raw[HD / 16];
#pragma unroll
    for (int kk = 0; kk < HD / 16; ++kk) raw[kk] = *reinterpret_cast<const u32x4*>(qrow + 16 * kk);
    // resolve the Q loads before the first DMA: inside the loop the compiler's wait for them
    // would be a vmcnt(0) that drains the ring
#pragma unroll
    for (int kk = 0; kk < HD / 16; ++kk) {
      asm volatile("" : "+v"(raw[kk]));
      bq[kk] = __builtin_bit_cast(bf16x8, raw[kk]);
    }
  }
  __syncthreads();  // block ids staged
#pragma unroll
  for (int c = 0; c < NS - 1; ++c)
    if (c < nchunk) issue(c);

  // K operand addresses: S^T row m = col holds token t0(m) (tile u = 0; u = 1 is t0 + 32, the same
  // swizzle); 16-B chunk 2 kk + h of that row sits at slot (2 kk + h) ^ (t0 & 15), i.e. at byte
  // offset k_lane ^ (kk << 5) (2 kk and h are disjoint bits)
  const int t0 = 16 * (col >> 4) + 8 * ((col >> 2) & 1) + 4 * ((col >> 3) & 1) + (col & 3);
  const int k_lane = t0 * 256 + (((t0 & 15) ^ h) << 4);
  const int v_lane = KBYTES + col * 32 + (((h ^ (col >> 3)) & 1) << 4);

  f32x16 o[HD / 32];
#pragma unroll
  for (int dt = 0; dt < HD / 32; ++dt) o[dt] = f32x16{};
  float m = -INFINITY, lsum = 0.f;  // running max (log2 units, column-uniform), this lane's partial sum

  // chunk c's pieces landed and its successor's slot is free: wait + barrier, then the DMA of
  // chunk c + NS - 1 (every wave runs this for every chunk of the workgroup)
  auto sync = [&](int c) __attribute__((always_inline)) {
    const int ahead = min(NS - 2, nchunk - 1 - c);  // later chunks whose pieces may still fly
    if (ahead >= 2) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * P) : "memory");
    } else if (ahead == 1) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(P) : "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    __builtin_amdgcn_s_barrier();  // ... and every wave is past chunk c - 1: its slot is free
    asm volatile("" ::: "memory");
    if (c + NS - 1 < nchunk) issue(c + NS - 1);
  };
  auto slot_of = [&](int c) { return static_cast<const unsigned char*>(ring + (c % NS) * SLOT); };
  int c = 0;
  float t[32];
  // chunks every row of the wave sees in full, then the diagonal (and context-end) chunks --
  // causal mask, V past the context zeroed -- in loops of their own (no branch on O inside)
  for (; c < n_full; ++c) {
    sync(c);
    attn32_scores<false>(slot_of(c), k_lane, bq, scale_log2, 0, m, lsum, o, t);
    attn32_pv<false>(slot_of(c), v_lane, 0, t, lsum, o);
  }
  for (; c < w_chunks; ++c) {
    sync(c);
    attn32_scores<true>(slot_of(c), k_lane, bq, scale_log2, c * KC + 8 * h - pos_q, m, lsum, o, t);
    attn32_pv<true>(slot_of(c), v_lane, c * KC + 8 * h - ctx, t, lsum, o);
  }
  for (; c < nchunk; ++c) sync(c);  // chunks in the causal future of every row of this wave
  if (!active || row0 + col >= q_end) return;
  {
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(lsum), __float_as_uint(lsum), false, false);
    lsum = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
  }
  const float inv = lsum > 0.f ? 1.f / lsum : 0.f;
  bf16_t* orow = out + (static_cast<size_t>(row0 + col) * n_q + qh) * HD + 4 * h;
#pragma unroll
  for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
    for (int gq = 0; gq < 4; ++gq) {  // O^T rows d = 32 dt + 8 gq + 4 h + (0..3) of this lane's column
      typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
      bf16x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = static_cast<__bf16>(o[dt][4 * gq + i] * inv);  // v_cvt_pk_bf16_f32 (RNE)
      *reinterpret_cast<bf16x4*>(orow + 32 * dt + 8 * gq) = v;
    }
}

}  // namespace

// Split size for a decode batch.  Measured on MI355X (tools/bench_ops.py, Qwen3-14B
// geometry, ctx 1700): two 32-token chunks per wave with BOTH chunks' loads issued
// before the first MFMA (256-token items) stream 5.2-5.4 TB/s at B = 160-608, against
// 4.4-4.7 for one chunk per wave (128-token items) -- and halve the split partials the
// merge kernel reads.  (Looping a wave over chunks one at a time was slower: 2-2.6 TB/s.)
constexpr int DEC_CPW = 2;
BCG_API int bcg_decode_split_tokens(int B, int n_kv, int max_tokens) { return DEC_WAVES * CHUNK * DEC_CPW; }
// Partial slots per (row, head): a row's own splits + up to DEC_MAX_SHARED_SPLITS of the
// shared-prefix pass (engine/cascade.py keeps shared tokens / its split within it).
// Only calls with the cascade tables reserve the shared slots (cascade = 0: a plain decode keeps
// the combine kernel's 64-split limit for its own splits, i.e. 16384 tokens of context).
BCG_API int bcg_decode_max_splits(int max_tokens, int cascade) {
  const int split = DEC_WAVES * CHUNK * DEC_CPW, own = (max_tokens + split - 1) / split, most = 64 - (cascade ? DEC_MAX_SHARED_SPLITS : 0);
  // one more for a row that a range of the streamed kernel cuts off its beat (its ranges are longer than a split: at the limit of 64 it
  // needs fewer than the splits)
  return (own < most ? own + 1 : own) + (cascade ? DEC_MAX_SHARED_SPLITS : 0);
}
// Longest context a decode call supports (the combine kernel reads at most 64 splits per row).
BCG_API int bcg_decode_max_context(int cascade) {
  return (64 - (cascade ? DEC_MAX_SHARED_SPLITS : 0)) * DEC_WAVES * CHUNK * DEC_CPW;
}

// kv_fp8: the caches hold OCP e4m3fn bytes (scale 1) instead of bf16.
BCG_API int bcg_paged_attention_decode(const void* q, const void* k_cache, const void* v_cache, int layer,
                                       int num_blocks, int n_kv, const int* block_tables, int max_blocks,
                                       const int* seq_lens, int B, int n_q, int hd, int block_size,
                                       float scale, float* workspace, int max_splits, int split_tokens,
                                       void* out, int kv_fp8, const int* kv_begin, const int* split_base,
                                       const int* grp_rows, int grp_cap, const int* grp_desc, int max_groups,
                                       const int* items, const int* n_items, int max_items,
                                       int shared_split_tokens, hipStream_t stream) {
  if (block_size != BS || n_q % n_kv || n_q / n_kv > 16 || B <= 0 || B > DEC_MAX_B) return -2;
  // with the cascade a row's own splits start after its shared tokens, in the slots after the
  // shared splits: the host sizes max_splits for both (bcg_decode_max_splits)
  const int own_slots = max_splits - (kv_begin ? DEC_MAX_SHARED_SPLITS : 0);
  if (split_tokens != DEC_WAVES * CHUNK * DEC_CPW || own_slots * split_tokens < max_blocks * BS) return -3;
  if (max_splits > 64) return -3;  // decode_combine_kernel: one lane per split
  Cascade cas{kv_begin, split_base, grp_rows, grp_cap, grp_desc, max_groups, items, n_items, max_items,
              shared_split_tokens};
  if (kv_begin && (!split_base || !grp_rows || !grp_desc || !items || !n_items || grp_cap < 0 || max_groups < 0 ||
                   max_items < 0 || shared_split_tokens <= 0 || shared_split_tokens % CHUNK))
    return -4;
  if (!kv_begin) cas = Cascade{nullptr, nullptr, nullptr, 0, nullptr, 0, nullptr, nullptr, 0, CHUNK};
  KVGeom g{static_cast<const bf16_t*>(k_cache), static_cast<const bf16_t*>(v_cache), layer, num_blocks, n_kv};
  const bf16_t* qb = static_cast<const bf16_t*>(q);
  bf16_t* ob = static_cast<bf16_t*>(out);
  const float sl = scale * LOG2E;
  if (hd == 128 && kv_fp8) {
    launch_decode<128, true, DEC_CPW>(qb, g, block_tables, max_blocks, seq_lens, B, n_q, sl, workspace,
                                             max_splits, ob, cas, stream);
  } else if (hd == 128) {
    launch_decode<128, false, DEC_CPW>(qb, g, block_tables, max_blocks, seq_lens, B, n_q, sl, workspace,
                                              max_splits, ob, cas, stream);
  } else if (hd == 64 && kv_fp8) {
    launch_decode<64, true, DEC_CPW>(qb, g, block_tables, max_blocks, seq_lens, B, n_q, sl, workspace,
                                            max_splits, ob, cas, stream);
  } else if (hd == 64) {
    launch_decode<64, false, DEC_CPW>(qb, g, block_tables, max_blocks, seq_lens, B, n_q, sl, workspace,
                                             max_splits, ob, cas, stream);
  } else {
    return -2;
  }
  return BCG_CHECK_LAUNCH();
}

// Rotary embedding, cache write and attention of a decode step (decode_pair_kernel): qkv [B, n_q + 2 n_kv, hd] as projected, one new token per row
// at `slots`; bf16 caches, hd 64 or 128.  parts, one, each, ways, extra: the rule by which several workgroups take a pair of a long row (PartRule; extra >= the parts
// beyond a pair's first that the rule can make: ways or B n_kv (parts - 1), each 0: the latter); workspace: 2 extra n_q / n_kv (hd + 2) floats, counters: `extra` zeros,
// left zero; of none null.  order: of the rows over the launch, a permutation (bcg_decode_order), or null.
BCG_API int bcg_decode_pairs(const void* qkv, const int* positions, const int* slots, const void* q_norm, const void* k_norm,
                             const float* cos_sin, float eps, void* k_cache, void* v_cache, int layer, int num_blocks, int n_kv,
                             const int* block_tables, int max_blocks, const int* seq_lens, int B, int n_q, int hd, int block_size,
                             float scale, int parts, int one, int each, int ways, int extra, float* workspace, int* counters, void* out, const int* order,
                             hipStream_t stream) {
  if ((hd != 64 && hd != 128) || block_size != BS || n_kv <= 0 || n_q % n_kv || n_q / n_kv > 16 || B <= 0 || B > DEC_MAX_B || max_blocks <= 0) return -2;
  const int64_t most = static_cast<int64_t>(B) * n_kv * (parts - 1);
  if (parts < 1 || parts > 64 || one < 0 || each < 0 || extra < (each > 0 && most > ways ? ways : most) || extra > 1 << 16 || ways < 0 ||
      (extra > 0 && (!workspace || !counters)) || max_blocks * BS > bcg_decode_max_context(0)) return -3;
  const PartRule rule{parts, one, each, ways, extra};
  const KVGeom g{static_cast<const bf16_t*>(k_cache), static_cast<const bf16_t*>(v_cache), layer, num_blocks, n_kv};
  const FusedArgs fa{static_cast<const bf16_t*>(qkv), positions, slots, static_cast<const bf16_t*>(q_norm),
                     static_cast<const bf16_t*>(k_norm), cos_sin, eps};
  auto run = [&](auto hd_c, auto waves_c) {
    constexpr int HD = decltype(hd_c)::value, NW = decltype(waves_c)::value;
    hipLaunchKernelGGL((decode_pair_kernel<HD, NW>), dim3(B * n_kv + extra), dim3(64 * NW), 0, stream, g, block_tables, max_blocks, seq_lens, B,
                       n_q, scale * LOG2E, rule, workspace, counters, static_cast<bf16_t*>(out), fa, order);
  };
  const bool many = B * n_kv + (each == 0 ? extra : 0) > (hd == 64 ? 512 : 1024);   // (see Pair)
  using std::integral_constant;
  if (hd == 64)
    many ? run(integral_constant<int, 64>{}, integral_constant<int, 4>{}) : run(integral_constant<int, 64>{}, integral_constant<int, 8>{});
  else
    many ? run(integral_constant<int, 128>{}, integral_constant<int, 2>{}) : run(integral_constant<int, 128>{}, integral_constant<int, 4>{});
  return BCG_CHECK_LAUNCH();
}

// order [B] = the rows, longest context first
BCG_API int bcg_decode_order(const int* seq_lens, int B, int* order, hipStream_t stream) {
  if (B <= 0 || B > DEC_MAX_B) return -2;
  hipLaunchKernelGGL(decode_order_kernel, dim3((B + 63) / 64), dim3(256), 0, stream, seq_lens, B, order);
  return BCG_CHECK_LAUNCH();
}

// nt: 16-row query tiles per wave; only 4 is built (0 = default).
BCG_API int bcg_paged_attention_prefill(const void* q, const void* k_cache, const void* v_cache, int layer,
                                        int num_blocks, int n_kv, const int* block_tables, int max_blocks,
                                        const int* q_start, const int* seq_lens, const int* tiles, int n_tiles,
                                        int n_q, int hd, int block_size, float scale, void* out, int nt,
                                        int kv_fp8, hipStream_t stream) {
  if (block_size != BS || n_q % n_kv || n_tiles <= 0) return -2;
  KVGeom g{static_cast<const bf16_t*>(k_cache), static_cast<const bf16_t*>(v_cache), layer, num_blocks, n_kv};
  const float sl = scale * LOG2E;
  const bf16_t* qb = static_cast<const bf16_t*>(q);
  bf16_t* ob = static_cast<bf16_t*>(out);
  if (nt != 0 && nt != 4) return -2;
  if (hd == 128)
    kv_fp8 ? launch_prefill<128, true>(n_tiles, n_q, qb, g, block_tables, max_blocks, q_start, seq_lens, tiles, sl,
                                       ob, stream)
           : launch_prefill<128, false>(n_tiles, n_q, qb, g, block_tables, max_blocks, q_start, seq_lens, tiles, sl,
                                        ob, stream);
  else if (hd == 64)
    kv_fp8 ? launch_prefill<64, true>(n_tiles, n_q, qb, g, block_tables, max_blocks, q_start, seq_lens, tiles, sl,
                                      ob, stream)
           : launch_prefill<64, false>(n_tiles, n_q, qb, g, block_tables, max_blocks, q_start, seq_lens, tiles, sl,
                                       ob, stream);
  else
    return -2;
  return BCG_CHECK_LAUNCH();
}

// The 32x32 LDS-staged form (prefill_attn32_kernel): `tiles` holds tiles of at most tile_rows
// rows -- 128 (4 waves, 2-slot ring, two workgroups per CU) or 256 (8 waves, 3-slot ring).
// bf16 KV cache and head dim 128 only (-2 otherwise: the caller uses the 16x16 kernel).
constexpr int PREFILL32_NS4 = 2, PREFILL32_NS8 = 3;  // ring slots at 4 / 8 waves (LDS: 2 or 1 workgroups per CU)
BCG_API int bcg_paged_attention_prefill32(const void* q, const void* k_cache, const void* v_cache, int layer,
                                          int num_blocks, int n_kv, const int* block_tables, int max_blocks,
                                          const int* q_start, const int* seq_lens, const int* tiles, int n_tiles,
                                          int n_q, int hd, int block_size, float scale, void* out, int tile_rows,
                                          int kv_fp8, hipStream_t stream) {
  if (block_size != BS || n_kv <= 0 || n_q % n_kv || n_tiles <= 0 || n_q > 65535 || hd != 128 || kv_fp8 ||
      max_blocks > PREFILL32_MAX_BLOCKS || static_cast<long long>(n_tiles) * n_q > 0x7fffffffLL)
    return -2;
  KVGeom g{static_cast<const bf16_t*>(k_cache), static_cast<const bf16_t*>(v_cache), layer, num_blocks, n_kv};
  const float sl = scale * LOG2E;
  const bf16_t* qb = static_cast<const bf16_t*>(q);
  bf16_t* ob = static_cast<bf16_t*>(out);
  const dim3 grid(n_tiles * n_q);  // XCD-grouped 1-D order (see the kernel)
  if (tile_rows == 128)
    hipLaunchKernelGGL((prefill_attn32_kernel<4, PREFILL32_NS4>), grid, dim3(256), 0, stream, qb, g, block_tables,
                       max_blocks, q_start, seq_lens, tiles, n_q, sl, ob, n_tiles);
  else if (tile_rows == 256)
    hipLaunchKernelGGL((prefill_attn32_kernel<8, PREFILL32_NS8>), grid, dim3(512), 0, stream, qb, g, block_tables,
                       max_blocks, q_start, seq_lens, tiles, n_q, sl, ob, n_tiles);
  else
    return -2;
  return BCG_CHECK_LAUNCH();
}
