// Recurrence with one decay per head over chunks of tokens (retention, scalar-decay state spaces; long segments):
//
//   S_t = g_t S_(t-1) + b_t k_t v_t^T,  o_t = S_t^T q_t        S fp32 [dim, vdim] per head, g in [0, 1]
//
// (g the same for every token or one number per token; b = 1 or one number per token).  A chunk of CT tokens is one
// set of matrix products instead of CT steps; with S the state in front of the chunk and
// W(r, s) = g_(s + 1) ... g_r the decay from token s of the chunk to token r,
//
//   o_r = (g_0 ... g_r) S^T q_r + sum_(s <= r) W(r, s) b_s (q_r . k_s) v_s
//   S  <- (g_0 ... g_n-1) S + sum_s W(n - 1, s) b_s k_s v_s^T            (n tokens in the chunk)
//
// Everything is fp32 (true-fp32 MFMAs, `mma16`); v is read in the activation type T.  Every W is a product of decays (in
// double, rounded once), never a quotient (a decay of 0 cuts cleanly): inside a 16-token block directly, across blocks as (from s to the end of
// its block) x (whole blocks) x (from the start of r's block to r).  The token-by-token form of seqmix_state.hip serves
// short segments; both leave the same state up to rounding.
//
// Two launches.  scores_kernel computes the q_r . k_s of all chunks at once (heads that share q and k
// share them, and so do the workgroups of a head).  chunk_kernel walks a segment's chunks:
// one workgroup per (segment, head, VT value columns), four waves.  The chunk's values lie in LDS transposed, and so does
// the state (value column by value column).  Wave w owns the chunk's queries 16 w .. 16 w + 15
// and the state's key features from 16 ND w on (a lane's ND features are neighbours).  The products are
// arranged so that a result in C registers is the next product's B operand (no shuffle):
//   S^T Q^T       [value column x query]   from the state in LDS
//   V^T (K Q^T)   [value column x query]   scores weighted by W b, added to it
//   V^T K         [value column x key feature], keys weighted by W b: the state's update
// The walk is a serial chain, so its operands are fetched a chunk ahead into the registers that the phase before has
// just used up (no wave needs another wave's keys or queries: they do not pass LDS), and VT shrinks where the launch would leave CUs
// idle.  What bounds it: the fp32 matrix rate (32 cycles per 16 x 16 x 4) where all CUs are busy, else the chain; of a chunk's 9500 cycles
// in workgroups of 16 columns 2900 are the state's update, 2300 the scores' products, 1500 the old state's, 1400 staging.  A chunk's
// decays are made once, by two waves, and read by all; no load stands behind a branch.  Measured, both launches, before and now:
// 3 segments of 700 tokens, 8 heads, 128 x 256 states: 91 -> 82 us; 64 heads of 128 x 128 that share keys: 8 segments of 1000 502 -> 465 (token by
// token: 1552; the matrix rate alone: 250), 8 segments of 600 to 1400 540 -> 510, 24 of 300 469 -> 441, one of 2000 207 -> 181.  Adding up the states
// of all chunks at once, carrying them along and reading them in three more launches: 73 us in the first case, up to twice as long in the others.
// Rounding, against float64 (relative rms, token by token -> here): decays about 0.5: 8.4e-8 -> 7.4e-8, 0.9: 1.1e-7 -> 1.0e-7, 0.99:
// 2.5e-7 -> 1.2e-7, 0.999: 4.6e-7 -> 1.5e-7.  That takes the scores in double (parallel, so nearly free), decay products in
// double, and short chains in the fp32 accumulators (one chain over all features and keys: 1.5e-7 at decays about 0.5).
#include <algorithm>
#include <type_traits>

#include "seqmix_common.h"

namespace {

constexpr int CT = 64, NTH = 256;

struct ChunkArgs {
  const float* q; const float* k;                   // [T, Gq, dim]
  const float* g; int g_token;                      // [H] (g_token 0) or [T, H]
  const float* beta;                                // [T, H] or null
  const void* v; int64_t v_stride;                  // [T, >= H vdim]
  const int* positions; const int* q_start; const int* state_rows;
  float* state;                                     // [n_rows, H, dim, vdim]
  float* out;                                       // [T, H, vdim]
  float* scores;                                    // [chunks, Gq, CT (query), CT (key)]
  int n_rows, B, H, Gq, dim, vdim, vec;             // vec: rows of q / k are 16-byte aligned
  int min_len;                                      // shorter segments are the token-by-token kernel's
};

// Segment b's chunk c has the number q_start[b] / CT + b + c: at most T / CT + B numbers, no two chunks alike.
__device__ __forceinline__ int chunk_base(const int* q_start, int b) { return q_start[b] / CT + b; }

// four fp32 at p[0..3], zero from n_valid on
__device__ __forceinline__ f32x4 load4(const float* p, int n_valid, bool vec) {
  f32x4 r = {0.f, 0.f, 0.f, 0.f};
  if (n_valid >= 4 && vec) return *reinterpret_cast<const f32x4*>(p);
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (j < n_valid) r[j] = p[j];
  return r;
}

// FULL: whole aligned tiles (dim = 16 DC): no branch around a load
template <bool FULL>
__device__ __forceinline__ f32x4 load4f(const float* p, int n_valid, bool vec) {
  if constexpr (FULL) return *reinterpret_cast<const f32x4*>(p);
  else return load4(p, n_valid, vec);
}

template <int DC, bool FULL>
__global__ __launch_bounds__(NTH) void scores_kernel(ChunkArgs a) {
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), col = lane & 15, grp = lane >> 4;
  const int id = blockIdx.x, gq = blockIdx.y, dim = a.dim;
  int lo = 0, hi = a.B - 1;   // the last segment whose first number is <= id
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (chunk_base(a.q_start, mid) <= id) lo = mid; else hi = mid - 1;
  }
  const int t0 = a.q_start[lo], t1 = a.q_start[lo + 1], first = t0 + (id - chunk_base(a.q_start, lo)) * CT;
  if (t1 - t0 < a.min_len || first < t0 || first >= t1) return;
  for (int e = wave; e < 10; e += 4) {   // the ten 16 x 16 tiles on and under the diagonal
    const int rt = e >= 6 ? 3 : e >= 3 ? 2 : e >= 1 ? 1 : 0, st = e - rt * (rt + 1) / 2;
    if (first + 16 * rt >= t1) continue;
    const float* qrow = a.q + (static_cast<size_t>(min(first + 16 * rt + col, t1 - 1)) * a.Gq + gq) * dim + 4 * grp;
    // (register i of a double result holds row grp + 4 i of the first operand: lane `col` supplies the key that makes it 4 grp + i)
    const int key = 4 * (col & 3) + (col >> 2);
    const float* krow = a.k + (static_cast<size_t>(min(first + 16 * st + key, t1 - 1)) * a.Gq + gq) * dim + 4 * grp;
    f32x4 qf[DC], kf[DC];
#pragma unroll
    for (int c = 0; c < DC; ++c) {
      qf[c] = load4f<FULL>(qrow + 16 * c, dim - 16 * c - 4 * grp, a.vec);
      kf[c] = load4f<FULL>(krow + 16 * c, dim - 16 * c - 4 * grp, a.vec);
    }
    typedef double f64x4 __attribute__((ext_vector_type(4)));
    f64x4 s = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int c = 0; c < DC; ++c)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        s = __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>(kf[c][j]), static_cast<double>(qf[c][j]), s, 0, 0, 0);
    f32x4 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = s[i];
    *reinterpret_cast<f32x4*>(a.scores + ((static_cast<size_t>(id) * a.Gq + gq) * CT + 16 * rt + col) * CT + 16 * st + 4 * grp) = r;
  }
}

// the value N lanes away in the row of 16 (1 from outside it)
template <int CTRL>
__device__ __forceinline__ double row_move(double x) {
  const int lo = __builtin_amdgcn_update_dpp(__double2loint(1.0), __double2loint(x), CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(__double2hiint(1.0), __double2hiint(x), CTRL, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}
template <int CTRL>
__device__ __forceinline__ double row_mul(double x) { return x * row_move<CTRL>(x); }

// DC: 16-wide tiles of key features (dim <= 16 DC).
template <typename T, int DC, int VT, bool FULL>
__global__ __launch_bounds__(NTH, DC <= 8 ? 2 : 1) void chunk_kernel(ChunkArgs a) {
  typedef typename Elem<T>::frag F;
  constexpr int LDK = 16 * DC + 4, LDV = CT + 4, ND = (DC + 3) / 4, NU = VT / 16;
  __shared__ __attribute__((aligned(16))) float Ss[VT * LDK];   // [value column][feature]
  __shared__ __attribute__((aligned(16))) T Vs[VT * LDV];       // [value column][token]
  __shared__ __attribute__((aligned(16))) float gs[CT], bs[CT];
  __shared__ double pre[CT], post[CT], whole[4];   // decay from a block's start to the token; that behind the token, times b; over a block
  __shared__ __attribute__((aligned(16))) float front[CT], tail[CT];   // decay from the chunk's start to the token; that to its end behind the token, times b
  __shared__ int wild;   // some value was infinite or NaN: it must not reach earlier queries as 0 x value
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), col = lane & 15, grp = lane >> 4;
  int b = blockIdx.x, h = blockIdx.y;
  if constexpr (VT == 64) segment_of(a.q_start, a.B, false, b, h);   // (fewer columns: fewer workgroups than places, where the order costs 2 to 3 us)
  const int v0 = blockIdx.z * VT;
  const int t0 = a.q_start[b], t1 = a.q_start[b + 1], sr = a.state_rows[b];
  if (t1 - t0 < a.min_len || sr < 0 || sr >= a.n_rows) return;
  const int gq = h / (a.H / a.Gq), dim = a.dim, vdim = a.vdim;
  float* Sg = a.state + (static_cast<size_t>(sr) * a.H + h) * dim * vdim + v0;
  const bool carry = a.positions[t0] != 0;
  const bool vec_s = (vdim & 3) == 0;
  const int d0 = 16 * ND * wave + ND * col;   // this lane's features of the state: d0 .. d0 + ND - 1
  constexpr bool OWNERS = FULL && DC % 4 == 0;   // every wave has features (of 32, two waves have none: they must not read past a row)
  const bool vec_k = OWNERS || (ND > 1 && a.vec && (dim & 3) == 0 && d0 + ND <= dim);
  f32x4 S[ND][NU];   // lane: S^T[value column 16 u + 4 grp + i][feature d0 + m]
#pragma unroll
  for (int m = 0; m < ND; ++m)
#pragma unroll
    for (int u = 0; u < NU; ++u)
      S[m][u] = (carry && d0 + m < dim) ? load4(Sg + static_cast<size_t>(d0 + m) * vdim + 16 * u + 4 * grp, vdim - v0 - 16 * u - 4 * grp, vec_s)
                                        : f32x4{0.f, 0.f, 0.f, 0.f};
  const bool owner = 16 * ND * wave < dim;   // (wave-uniform) the wave has features
  const int place = 16 * wave + col;         // this lane's query in a chunk

  // ---- loads, one chunk ahead; rows past the segment repeat its last one and are masked where they are used.  No branch around a load (the last
  // chunk loads itself again): behind one hipcc waits for every load in flight, the youngest too ----
  f32x4 qf[DC];
  float kf[4][4][ND];
  f32x4 rf[4];
  uint32_t vf[NU][4];   // (bits; packed where they are staged: packing waits for the loads)
  float gf, bf;
  const T* vbase = static_cast<const T*>(a.v) + static_cast<size_t>(h) * vdim + v0;
  const int v_col = tid % VT, v_tok = 4 * (tid / VT);
  const uint32_t v_src = min(v_col, vdim - 1 - v0);   // (columns past the state repeat its last one and are not stored)
  // (a chunk's rows start at a uniform address; a lane's place in the chunk is a 32-bit offset)
  const uint32_t row = static_cast<uint32_t>(a.Gq) * dim, v_row = static_cast<uint32_t>(a.v_stride);
  auto at = [](const auto* base, uint32_t o) {   // (32 bits of bytes: one register beside a uniform base)
    typedef std::remove_pointer_t<decltype(base)> E;
    return reinterpret_cast<E*>(reinterpret_cast<const char*>(base) + static_cast<uint32_t>(o * sizeof(E)));
  };
  const float* betas = a.beta != nullptr ? a.beta : a.g;
  const size_t beta_token = a.beta != nullptr ? a.H : a.g_token;
  auto load_q = [&](int first) {
    const float* base = a.q + static_cast<size_t>(first) * row + gq * dim;
    const uint32_t o = min(place, t1 - 1 - first) * row + 4 * grp;
#pragma unroll
    for (int c = 0; c < DC; ++c) qf[c] = load4f<FULL>(at(base, o + 16 * c), dim - 16 * c - 4 * grp, a.vec);
  };
  auto load_k = [&](int first, int tt) {
    const float* base = a.k + static_cast<size_t>(first) * row + gq * dim;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t o = min(16 * tt + 4 * grp + j, t1 - 1 - first) * row + d0;
      if constexpr (ND > 1) {
        typedef float fv __attribute__((ext_vector_type(ND)));
        if (vec_k) {
          const fv x = *reinterpret_cast<const fv*>(at(base, o));
#pragma unroll
          for (int m = 0; m < ND; ++m) kf[tt][j][m] = x[m];
          continue;
        }
      }
#pragma unroll
      for (int m = 0; m < ND; ++m) kf[tt][j][m] = OWNERS || d0 + m < dim ? *at(base, o + m) : 0.f;
    }
  };
  auto load_r = [&](int first, int id) {
    const float* base = a.scores + (static_cast<size_t>(id) * a.Gq + gq) * CT * CT;
    const uint32_t o = place * CT + 4 * grp;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
      rf[kt] = *reinterpret_cast<const f32x4*>(at(base, o + 16 * min(kt, wave)));
  };
  auto load_v = [&](int first) {
    const T* base = vbase + static_cast<size_t>(first) * a.v_stride;
#pragma unroll
    for (int p = 0; p < NU; ++p)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const T x = *at(base, min(v_tok + p * (4 * NTH / VT) + j, t1 - 1 - first) * v_row + v_src);
        if constexpr (sizeof(T) == 2) vf[p][j] = x; else vf[p][j] = __float_as_uint(x);
      }
    const size_t t = min(first + lane, t1 - 1);
    gf = a.g[t * a.g_token + h];
    bf = betas[t * beta_token + h];
  };
  auto value_frag = [&](int u, int tok) {   // V^T[value column 16 u + col][tokens tok .. tok + 3] as fp32
    const F f = *reinterpret_cast<const F*>(&Vs[(16 * u + col) * LDV + tok]);
    f32x4 r;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (sizeof(T) == 2) r[j] = bf2f(static_cast<bf16_t>(f[j])); else r[j] = f[j];
    }
    return r;
  };
  if (tid == 0) wild = 0;
  __syncthreads();
  int id = chunk_base(a.q_start, b);
  load_v(t0);
  load_q(t0);
  load_r(t0, id);
#pragma unroll
  for (int tt = 0; tt < 4; ++tt) load_k(t0, tt);
  for (int first = t0; first < t1; first += CT, ++id) {
    const int n = min(CT, t1 - first);
    const int ahead = first + CT < t1 ? first + CT : first, id_ahead = first + CT < t1 ? id + 1 : id;
    // ---- values, state and decays to LDS ----
#pragma unroll
    for (int p = 0; p < NU; ++p) {
      F f;
      bool odd = false;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t x = first + v_tok + p * (4 * NTH / VT) + j < t1 ? vf[p][j] : 0u;
        if constexpr (sizeof(T) == 2) { f[j] = static_cast<short>(x); odd |= (x & 0x7F80u) == 0x7F80u; }
        else { f[j] = __uint_as_float(x); odd |= (x & 0x7F800000u) == 0x7F800000u; }
      }
      *reinterpret_cast<F*>(&Vs[v_col * LDV + v_tok + p * (4 * NTH / VT)]) = f;
      if (odd) wild = 1;
    }
    if (ND * wave < DC) {   // every column of the tiles: what lies past dim is zero, and multiplied
#pragma unroll
      for (int u = 0; u < NU; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int m = 0; m < ND; ++m)
            if (DC % 4 == 0 || d0 + m < 16 * DC) Ss[(16 * u + 4 * grp + i) * LDK + d0 + m] = S[m][u][i];
    }
    if (wave <= 1) {   // lane = token
      const bool in = first + lane < t1;
      gf = in ? gf : 1.0f;
      bf = in ? (a.beta != nullptr ? bf : 1.0f) : 0.0f;
      const double p = row_mul<0x118>(row_mul<0x114>(row_mul<0x112>(row_mul<0x111>(static_cast<double>(gf)))));   // row_shr 1, 2, 4, 8
      auto block = [&](int k) {
        return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(p), 16 * k + 15), __builtin_amdgcn_readlane(__double2loint(p), 16 * k + 15));
      };
      if (wave == 0) {
        const double w0 = block(0), w1 = block(1), w2 = block(2);
        gs[lane] = gf;
        bs[lane] = bf;
        pre[lane] = p;
        front[lane] = p * (grp == 0 ? 1.0 : grp == 1 ? w0 : grp == 2 ? w0 * w1 : w0 * w1 * w2);
        if (col == 15) whole[grp] = p;
      } else {
        const double s = row_mul<0x108>(row_mul<0x104>(row_mul<0x102>(row_mul<0x101>(static_cast<double>(gf)))));   // row_shl 1, 2, 4, 8
        const double after = row_move<0x101>(s) * bf, w1 = block(1), w2 = block(2), w3 = block(3);
        post[lane] = after;
        tail[lane] = after * (grp == 3 ? 1.0 : grp == 2 ? w3 : grp == 1 ? w2 * w3 : w1 * w2 * w3);
      }
    }
    __syncthreads();
    load_v(ahead);
    const double wh[4] = {whole[0], whole[1], whole[2], whole[3]};
    // few columns: the walk's length counts and not its products: nothing of a chunk stands behind a branch, so one step's reads and weights
    // fly under the products of the one before (blocks of keys that a wave does not see have weights of zero)
    constexpr bool FEW = VT == 16;
    f32x4 o[NU];
#pragma unroll
    for (int u = 0; u < NU; ++u) o[u] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (FEW || 16 * wave < n) {
      const double here = pre[place];
#pragma unroll
      for (int kt = 0; kt < 3; ++kt) {   // the blocks before the queries' own
        if (FEW || kt < wave) {   // (wave-uniform)
          double g = here;
#pragma unroll
          for (int k = 1; k < 3; ++k) g *= k > kt && k < wave ? wh[k] : 1.0;
          f32x4 s;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            s[i] = rf[kt][i] * static_cast<float>(post[16 * kt + 4 * grp + i] * g);
            if (FEW && kt >= wave) s[i] = 0.f;
          }
#pragma unroll
          for (int u = 0; u < NU; ++u) {
            f32x4 x = value_frag(u, 16 * kt + 4 * grp);
            if (FEW && kt >= wave) x = f32x4{0.f, 0.f, 0.f, 0.f};   // (a later value may be infinite)
            o[u] += mma16(x, s, f32x4{0.f, 0.f, 0.f, 0.f});
          }
        }
      }
      // their own: the decay over tokens key + 1 .. query of the block
      f32x4 s = wave == 0 ? rf[0] : wave == 1 ? rf[1] : wave == 2 ? rf[2] : rf[3];
      {
        // (a product along the lanes of a row: lane = token)
        double x = row_mul<0x118>(row_mul<0x114>(row_mul<0x112>(row_mul<0x111>(static_cast<double>(col >= 4 * grp + 4 ? gs[16 * wave + col] : 1.0f)))));
        const f32x4 own = *reinterpret_cast<const f32x4*>(&gs[16 * wave + 4 * grp]);
        const f32x4 be = *reinterpret_cast<const f32x4*>(&bs[16 * wave + 4 * grp]);
#pragma unroll
        for (int i = 3; i >= 0; --i) {
          s[i] = 4 * grp + i <= col ? s[i] * (x * be[i]) : 0.f;
          x *= static_cast<double>(4 * grp + i <= col ? own[i] : 1.0f);
        }
      }
      if (!wild) {
#pragma unroll
        for (int u = 0; u < NU; ++u) o[u] += mma16(value_frag(u, 16 * wave + 4 * grp), s, f32x4{0.f, 0.f, 0.f, 0.f});
      } else {   // (rare) key by key, masked
#pragma unroll 1
        for (int key = 0; key < 16; ++key) {
          const float x = __shfl((key & 2) ? ((key & 1) ? s[3] : s[2]) : ((key & 1) ? s[1] : s[0]), (key >> 2) * 16 + col, 64);
#pragma unroll
          for (int u = 0; u < NU; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const float y = o[u][i] + x * Elem<T>::ld(Vs[(16 * u + 4 * grp + i) * LDV + 16 * wave + key]);
              o[u][i] = key <= col ? y : o[u][i];
            }
        }
      }
    }
    load_r(ahead, id_ahead);
    if (FEW || 16 * wave < n) {
      if (carry || first > t0) {   // S^T Q^T, in chains of one feature tile (one long chain rounds twice as much)
        const float g = front[place];
#pragma unroll
        for (int u = 0; u < NU; ++u)
#pragma unroll
          for (int c = 0; c < DC; ++c)
            o[u] += g * mma16(*reinterpret_cast<const f32x4*>(&Ss[(16 * u + col) * LDK + 16 * c + 4 * grp]), qf[c], f32x4{0.f, 0.f, 0.f, 0.f});
      }
      if (place < n) {
        float* orow = a.out + (static_cast<size_t>(first + place) * a.H + h) * vdim + v0;
#pragma unroll
        for (int u = 0; u < NU; ++u) {
          const int e = 16 * u + 4 * grp;
          if (vec_s && v0 + e + 3 < vdim) {
            *reinterpret_cast<f32x4*>(orow + e) = o[u];
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (v0 + e + i < vdim) orow[e + i] = o[u][i];
          }
        }
      }
    }
    load_q(ahead);
    // ---- the state behind the chunk ----
    if (OWNERS || owner) {
      if (n < CT) {   // (no key past the segment, not even against a weight of zero: it may be infinite)
#pragma unroll
        for (int tt = 0; tt < 4; ++tt)
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int m = 0; m < ND; ++m) kf[tt][j][m] = 16 * tt + 4 * grp + j < n ? kf[tt][j][m] : 0.f;
      }
      const float gn = (wh[0] * wh[1]) * (wh[2] * wh[3]);
#pragma unroll
      for (int m = 0; m < ND; ++m)
#pragma unroll
        for (int u = 0; u < NU; ++u) S[m][u] *= gn;
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) {
        if (FEW || 16 * tt < n) {   // (uniform)
          const f32x4 w = *reinterpret_cast<const f32x4*>(&tail[16 * tt + 4 * grp]);
          f32x4 x[NU];
#pragma unroll
          for (int u = 0; u < NU; ++u) x[u] = value_frag(u, 16 * tt + 4 * grp);
#pragma unroll
          for (int m = 0; m < ND; ++m) {
            f32x4 kw;
#pragma unroll
            for (int j = 0; j < 4; ++j) kw[j] = kf[tt][j][m] * w[j];
#pragma unroll
            for (int u = 0; u < NU; ++u) S[m][u] += mma16(x[u], kw, f32x4{0.f, 0.f, 0.f, 0.f});
          }
        }
        load_k(ahead, tt);
      }
    }
    __syncthreads();   // every reader of the chunk and of the old state is done
  }
#pragma unroll
  for (int m = 0; m < ND; ++m) {
    if (d0 + m >= dim) continue;
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int e = 16 * u + 4 * grp;
      float* p = Sg + static_cast<size_t>(d0 + m) * vdim + e;
      if (vec_s && v0 + e + 3 < vdim) {
        *reinterpret_cast<f32x4*>(p) = S[m][u];
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (v0 + e + i < vdim) p[i] = S[m][u][i];
      }
    }
  }
}

template <typename T, int DC, bool FULL>
int launch_chunks(const ChunkArgs& a, int n_chunks, hipStream_t s) {
  scores_kernel<DC, FULL><<<dim3(n_chunks, a.Gq), NTH, 0, s>>>(a);
  // Value columns per workgroup: 16 while these keep to two workgroups per CU, the walk is serial and idle CUs cost nothing (3 segments of 700,
  // 8 heads of 128 x 256: 16 columns 83 us, 32 88, 64 139; one of 2000, 64 heads of 128 x 128: 181, 185, 313); 32 up to two workgroups per CU, of keys
  // wider than 64 up to three (6 segments of 700: 16 columns 166, 32 131, 64 163; 3 of 2000: 507, 415, 450; 64 of 200, 4 heads of 64 x 64: 54, 46, 52); 64
  // past them (4 of 2000: 672, 501, 458; 100 of 200: 77, 68, 60).
  const int64_t wide = static_cast<int64_t>(a.B) * a.H * ((a.vdim + 63) / 64);
  if (wide > (DC > 4 ? 384 : 256)) chunk_kernel<T, DC, 64, FULL><<<segment_grid(a.H, a.B, (a.vdim + 63) / 64), NTH, 0, s>>>(a);
  else if (wide > 128) chunk_kernel<T, DC, 32, FULL><<<dim3(a.B, a.H, (a.vdim + 31) / 32), NTH, 0, s>>>(a);
  else chunk_kernel<T, DC, 16, FULL><<<dim3(a.B, a.H, (a.vdim + 15) / 16), NTH, 0, s>>>(a);
  return BCG_CHECK_LAUNCH();
}

template <typename T, int DC>
int launch_full(const ChunkArgs& a, int n_chunks, hipStream_t s) {
  if constexpr (sizeof(T) == 2) {
    if (a.vec && a.dim == 16 * DC) return launch_chunks<T, DC, true>(a, n_chunks, s);
  }
  return launch_chunks<T, DC, false>(a, n_chunks, s);
}

template <typename T>
int launch_dim(const ChunkArgs& a, int n_chunks, hipStream_t s) {
  if (a.dim <= 32) return launch_full<T, 2>(a, n_chunks, s);
  if (a.dim <= 64) return launch_full<T, 4>(a, n_chunks, s);
  if (a.dim <= 128) return launch_full<T, 8>(a, n_chunks, s);
  return launch_full<T, 16>(a, n_chunks, s);
}

}  // namespace

// `scores` takes (T / tokens + B) Gq tokens^2 fp32 elements
BCG_API int bcg_decay_chunks_tokens() { return CT; }

// g: [H] (g_token 0) or [T, H] (g_token H); beta [T, H] or null.  Segments of fewer than `min_len` tokens are left alone.
BCG_API int bcg_decay_chunks(const void* q32, const void* k32, const void* g, int g_token, const void* beta, const void* v,
                             int64_t v_stride, const void* positions, const void* q_start, const void* state_rows, void* state,
                             int n_rows, void* out, void* scores, int T_, int B, int H, int Gq, int dim, int vdim, int min_len,
                             int is_f32, void* stream) {
  if (B <= 0 || T_ <= 0) return 0;
  if (dim < 1 || dim > 256 || vdim < 1 || H <= 0 || Gq <= 0 || H % Gq || H > 65535 || (vdim + 15) / 16 > 65535 || min_len < 1) return -2;
  auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  if (!al16(state) || !al16(out) || !al16(scores) || scores == nullptr || (g_token != 0 && g_token != H)) return -2;
  ChunkArgs a;
  a.q = static_cast<const float*>(q32); a.k = static_cast<const float*>(k32);
  a.g = static_cast<const float*>(g); a.g_token = g_token; a.beta = static_cast<const float*>(beta);
  a.v = v; a.v_stride = v_stride;
  a.positions = static_cast<const int*>(positions); a.q_start = static_cast<const int*>(q_start);
  a.state_rows = static_cast<const int*>(state_rows);
  a.state = static_cast<float*>(state); a.out = static_cast<float*>(out); a.scores = static_cast<float*>(scores);
  a.n_rows = n_rows; a.B = B; a.H = H; a.Gq = Gq; a.dim = dim; a.vdim = vdim;
  a.vec = dim % 4 == 0 && al16(q32) && al16(k32);
  a.min_len = min_len;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return is_f32 ? launch_dim<float>(a, T_ / CT + B, s) : launch_dim<bf16_t>(a, T_ / CT + B, s);
}
