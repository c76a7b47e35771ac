// Device-side building blocks of the adapter-indexed LoRA delta, shared by the stand-alone gather-matmul
// kernels and by the decode kernels that carry LoRA work inside their own launch.
#pragma once
#include "common.h"

constexpr int LORA_KCHUNK = 512;   // K elements one wave covers per pass: 64 lanes x 8 fp16
constexpr int LORA_MAX_KC = 8;     // K-slices (fp32 partials) per token
constexpr int LORA_MAX_PROJ = 3;   // projections that share x in one batched shrink (q, k, v)
constexpr int LORA_MAX_KQ = 4;     // K-range blocks of dense shrink results

struct LoraKSplit { int ci; int kc; };

static inline LoraKSplit lora_k_split(int K) {
  int ci = ceil_div(K, LORA_KCHUNK * LORA_MAX_KC);
  if (ci < 1) ci = 1;
  return {ci, ceil_div(K, LORA_KCHUNK * ci)};
}

// A batch of shrink problems that share x and the token->adapter table:
//   v_part[p][c][t][:] = A[p][id_t][:, slice c] . x[t, slice c]        (fp32, one partial per K-slice c)
struct LoraShrinkBatch {
  const f16* A[LORA_MAX_PROJ];   // [n_ad, r, K] each
  int n_proj;
  float* vpart;                  // [n_proj][kc][T][r]
  const f16* x;
  const int32_t* ids;
  int T, K, r, n_ad, ci, kc, frag_tt;
  int speculate;                 // request A before the adapter table is read (adapters expected to be in use)
  const int32_t* bucket_of;      // optional [T]: rank bucket of each token; tokens of other buckets count as unadapted
  int bucket;
};

// Adapter id of token t as this launch sees it: -1 outside the table and for tokens of another rank bucket.
__device__ __forceinline__ int lora_token_id(const int32_t* __restrict__ ids, const int32_t* __restrict__ bucket_of,
                                             int bucket, int t, int T) {
  if (t >= T) return -1;
  if (bucket_of != nullptr && bucket_of[t] != bucket) return -1;
  return ids[t];
}

static inline int lora_shrink_units(const LoraShrinkBatch& b) { return b.n_proj * b.n_ad * b.kc; }

// Reduce G per-lane partials across the 64 lanes.  On return every lane holds in p[0] the full sum
// of partial index j (returned); lanes sharing j hold the same value.
template <int G>
__device__ __forceinline__ int reduce_transpose(float (&p)[G], int lane) {
  int j = 0;
  int off = 32;
#pragma unroll
  for (int n = G; n > 1; n >>= 1) {
    const int half = n >> 1;
    const bool hi = (lane & off) != 0;
#pragma unroll
    for (int i = 0; i < half; ++i) {
      // The two candidates are pinned in registers of their own (empty asm): left to itself the compiler folds the
      // selects of all levels into one dynamically indexed read of p[], which it lowers to a 16-way compare/select
      // chain per element - hundreds of instructions instead of two.
      float a = p[i], b = p[i + half];
      asm volatile("" : "+v"(a), "+v"(b));
      const float send = hi ? a : b;
      const float keep = hi ? b : a;
      p[i] = keep + __shfl_xor(send, off, WAVE);
    }
    j += hi ? half : 0;
    off >>= 1;
  }
#pragma unroll
  for (; off > 0; off >>= 1) p[0] += __shfl_xor(p[0], off, WAVE);
  return j;
}

// One wave: adapter a of projection p, K-slice c.  The first 16 rows of its slice of A[a] are requested before the
// token->adapter table has been read (when `speculate` is set: adapters are expected to be in use), so the wave
// pays one memory round trip, not two, before it can start; that matters when the unit shares a launch with a
// bandwidth-saturating GEMV and every round trip queues behind the weight stream.  Tokens bound to a are found
// with ballots; A stays in registers across token pairs whenever the whole slice fits (r <= 16, one chunk).
__device__ __forceinline__ void lora_shrink_unit(const LoraShrinkBatch& b, int unit, int lane) {
  constexpr int G = 16, TB = 2;
  const int c = unit % b.kc;
  const int a = (unit / b.kc) % b.n_ad;
  const int pj = unit / (b.kc * b.n_ad);
  if (b.A[pj] == nullptr) return;   // projection slot not adapted
  const f16* __restrict__ A = b.A[pj] + (size_t)a * b.r * b.K;
  float* __restrict__ vp = b.vpart + ((size_t)pj * b.kc + c) * b.T * b.r;
  const int kbase = c * b.ci * LORA_KCHUNK + lane * 8;
  const bool resident = b.r <= G && b.ci == 1;   // the wave's whole slice of A fits the register file
  const f16x8 zero8 = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
  f16x8 areg[G];
  int id = lora_token_id(b.ids, b.bucket_of, b.bucket, lane, b.T);
  if (resident && b.speculate) {
#pragma unroll
    for (int j = 0; j < G; ++j) areg[j] = (j < b.r && kbase < b.K) ? ld8(A + (size_t)j * b.K + kbase) : zero8;
  }
  bool loaded = resident && b.speculate;
  for (int t0 = 0; t0 < b.T; t0 += WAVE) {
    if (t0 > 0) id = lora_token_id(b.ids, b.bucket_of, b.bucket, t0 + lane, b.T);
    unsigned long long mask = __ballot(id == a);
    if (mask && resident && !loaded) {
      loaded = true;
#pragma unroll
      for (int j = 0; j < G; ++j) areg[j] = (j < b.r && kbase < b.K) ? ld8(A + (size_t)j * b.K + kbase) : zero8;
    }
    while (mask) {
      int tt[TB];
#pragma unroll
      for (int u = 0; u < TB; ++u) {
        tt[u] = -1;
        if (mask) {
          tt[u] = t0 + __builtin_ctzll(mask);
          mask &= mask - 1;
        }
      }
      for (int jb = 0; jb < b.r; jb += G) {
        float p[TB][G];
#pragma unroll
        for (int u = 0; u < TB; ++u)
#pragma unroll
          for (int j = 0; j < G; ++j) p[u][j] = 0.f;
        for (int ci = 0; ci < b.ci; ++ci) {
          const int k = kbase + ci * LORA_KCHUNK;
          f16x8 xv[TB];
#pragma unroll
          for (int u = 0; u < TB; ++u) {
            const int t = tt[u] >= 0 ? tt[u] : tt[0];
            xv[u] = k < b.K ? ld8(b.x + (b.frag_tt ? frag_offset(t, k, b.frag_tt) : (size_t)t * b.K + k)) : zero8;
          }
          if (!resident) {
#pragma unroll
            for (int j = 0; j < G; ++j) areg[j] = (jb + j < b.r && k < b.K) ? ld8(A + (size_t)(jb + j) * b.K + k) : zero8;
          }
#pragma unroll
          for (int j = 0; j < G; ++j)
#pragma unroll
            for (int u = 0; u < TB; ++u) p[u][j] = dot8(areg[j], xv[u], p[u][j]);
        }
#pragma unroll
        for (int u = 0; u < TB; ++u) {
          const int j = reduce_transpose<G>(p[u], lane);
          if (tt[u] >= 0 && jb + j < b.r && (lane & (WAVE / G - 1)) == 0) vp[(size_t)tt[u] * b.r + jb + j] = p[u][0];
        }
      }
    }
  }
}

// v[j] = scaling * sum_c v_part[c][t][j] for one token, summed in slice order (the order every consumer uses,
// so fused and stand-alone expands agree bit for bit).
// The slices are requested together and then added one by one: as a loop over kc, every addition waited for its own
// load - up to eight dependent round trips in front of an expand.
__device__ __forceinline__ float lora_v(const float* __restrict__ vpart_proj, int kc, int T, int r, int t, int j, float scaling) {
  float part[LORA_MAX_KC];
#pragma unroll
  for (int c = 0; c < LORA_MAX_KC; ++c) part[c] = c < kc ? vpart_proj[((size_t)c * T + t) * r + j] : 0.f;
  float v = 0.f;
#pragma unroll
  for (int c = 0; c < LORA_MAX_KC; ++c)
    if (c < kc) v += part[c];
  return v * scaling;
}

// Where an expand finds v for (token t, projection slot p, adapter id):
//   kc > 0  : K-slice partials v_part[p][c][t][:]                    (written by the shrink units)
//   kc == 0 : dense shrink results v_all[q][t][(p * n_ad + id) * r + :]  (written by a GEMV over weight rows that have
//             the A tables of all adapters appended; the adapter is picked here, by index).  kq >= 1 blocks q hold
//             the partial sums of kq ranges of K, added here in range order.
struct LoraVSource {
  const float* v;
  int kc, T, n_ad, ld, kq;
};

__device__ __forceinline__ float lora_v_from(const LoraVSource& s, int slot, int id, int r, int t, int j, float scaling) {
  if (s.kc > 0) return lora_v(s.v + (size_t)slot * s.kc * s.T * r, s.kc, s.T, r, t, j, scaling);
  const float* __restrict__ p = s.v + (size_t)t * s.ld + ((size_t)slot * s.n_ad + id) * r + j;
  float part[LORA_MAX_KQ];
#pragma unroll
  for (int q = 0; q < LORA_MAX_KQ; ++q) part[q] = q == 0 || q < s.kq ? p[(size_t)q * s.T * s.ld] : 0.f;   // all blocks requested together
  float a = part[0];
#pragma unroll
  for (int q = 1; q < LORA_MAX_KQ; ++q)
    if (q < s.kq) a += part[q];
  return a * scaling;
}

// The same dot product in two halves, so that a caller can issue the row's loads before the v values are ready:
// lora_row_load fetches up to 8 groups of 8 (r <= 64), lora_row_dot_regs consumes them in lora_row_dot's order.
template <int NGMAX>
__device__ __forceinline__ void lora_row_load(const f16* __restrict__ brow, int r, f16x8 (&bv)[NGMAX]) {
  const int ng = r >> 3;
#pragma unroll
  for (int q = 0; q < NGMAX; ++q) {
    bv[q] = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
    if (q < ng) bv[q] = ld8(brow + q * 8);
  }
}

template <int NGMAX>
__device__ __forceinline__ float lora_row_dot_regs(const f16x8 (&bv)[NGMAX], const float* __restrict__ v, int r) {
  float g[8];                           // r <= 8 * NGMAX; groups past NGMAX are empty
  const int ng = r >> 3;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    float s = 0.f;
    if (q < NGMAX) {
      if (q < ng) {
#pragma unroll
        for (int e = 0; e < 8; ++e) s = fmaf((float)bv[q < NGMAX ? q : 0][e], v[q * 8 + e], s);
      }
    }
    g[q] = s;
  }
  if (ng > 4) {
    g[0] = g[0] + g[1]; g[1] = g[2] + g[3]; g[2] = g[4] + g[5]; g[3] = g[6] + g[7];
  }
  if (ng > 2) {
    g[0] = g[0] + g[1]; g[1] = g[2] + g[3];
  }
  if (ng > 1) g[0] = g[0] + g[1];
  return g[0];
}

// delta = B_row[0..r) . v[0..r) with the summation tree of the stand-alone expand kernel: an fma chain over each
// group of 8, then pairwise sums of neighbouring groups.
__device__ __forceinline__ float lora_row_dot(const f16* __restrict__ brow, const float* __restrict__ v, int r) {
  float g[8];
  const int ng = r >> 3;
  for (int q = 0; q < ng; ++q) {
    const f16x8 bv = ld8(brow + q * 8);
    float s = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) s = fmaf((float)bv[e], v[q * 8 + e], s);
    g[q] = s;
  }
  for (int n = ng; n > 1; n >>= 1)
    for (int q = 0; q < n / 2; ++q) g[q] = g[2 * q] + g[2 * q + 1];
  return g[0];
}

#ifndef MLORA_ELT_F32
// ---------------------------------------------------------------------------------------------
// The deltas of any mix of adapters in the accumulators of a linear, y = x . W^T + v . B[id]^T with v = scaling * (sum of the shrink's K ranges).  Projections
// are row ranges of the fused weight.
// ---------------------------------------------------------------------------------------------

// The second operand of mfma_16x16x32 with the bits of fp32: eight values of a column, scaled by a power of two that brings the largest of the column's 32 below
// 2^15, as three fp16 parts.  11 bits each, the last one's step 2^-24: whole fp32 values down to 2^-14 of the largest, and 2^-39 of it below that.  48 cycles of a
// SIMD a product, against 256 of the fp32 matrix instruction, and fewer roundings.  (Two parts of the values as they are keep 22 bits, nothing below 2^-24, and
// make NaN of what is beyond 65504.)
struct Col32 {
  eltx8 part[3];
  float back;                 // the inverse of the scale
};
__device__ __forceinline__ Col32 col32_of(const float (&f)[8]) {
  float m = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) m = fmaxf(m, fabsf(f[e]));
  m = fmaxf(m, __shfl_xor(m, 16, WAVE));                         // the other k-groups of the column
  m = fmaxf(m, __shfl_xor(m, 32, WAVE));
  const int ex = (int)(__float_as_uint(m) >> 23);                // biased; 255: an infinity, for which no part but the first is taken
  const int sx = 268 - ex < 253 ? 268 - ex : 253;
  const float scale = __uint_as_float((unsigned)sx << 23);
  Col32 c;
  c.back = __uint_as_float((unsigned)(254 - sx) << 23);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float x = f[e] * scale;
    c.part[0][e] = (elt)x;
    const float y = ex < 255 ? x - (float)c.part[0][e] : 0.f;
    c.part[1][e] = (elt)y;
    c.part[2][e] = (elt)(y - (float)c.part[1][e]);
  }
  return c;
}
__device__ __forceinline__ f32x4 mfma_16x16x32_col32(eltx8 a, const Col32& b, f32x4 c) {
  f32x4 d = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int p = 2; p >= 0; --p) d = mfma_16x16x32(a, b.part[p], d);
#pragma unroll
  for (int q = 0; q < 4; ++q) c[q] = fmaf(d[q], b.back, c[q]);
  return c;
}

constexpr int DELTA_RANGES = 4;                // K ranges of the shrink that are in flight together in registers
struct LinearDeltas {
  const elt* B[3];            // [n_ad][n_rows][r]
  int n_begin[3], n_rows[3];
  const float* v;             // [n_proj][ranges][T][r], rows of tokens without adapter not written
  const int32_t* ids;         // [T]: outside 0 .. n_ad - 1 no adapter
  float scaling;
  int n_proj, r, n_ad, ranges;
};

// acc [NN][TT]: 16-row tiles of W (row0: their first rows) x tiles of 16 tokens from t0 on, as mfma_16x16x32 leaves them; left: the ids of this lane's
// tokens (-1 past T).  A wave takes the adapters of these tokens in turn and of the rounds - an adapter, 32 ranks - every step-th (a power of two above one, or one);
// both operands come straight from memory.  A product's columns are tokens, so a lane keeps the sums of a round where its own token names the adapter, and
// its accumulators as they were otherwise: what an adapter's tables hold, infinities and NaN too, stays with its tokens.  (Without a branch: behind one the loads of
// a wave's tiles would go out one after the other, 137 tokens x 12288 x 4096 42 instead of 36 us.)  Which wave
// does a round follows the order of the adapters among the tokens; a token's one or two rounds are different waves', and half[j] says which of them
// this wave has done for the lane's token (-1: none), so that the caller can add them in an order that does not depend on the other tokens.
// V32: v with the bits of fp32 (up to 64 tokens); else as fp16 hi and lo halves.
template <int NN, int TT, bool V32>
__device__ __forceinline__ void linear_add_deltas(f32x4 (&acc)[NN][TT], const LinearDeltas& lo, int (&left)[TT], int (&half)[TT], int T, int t0, const int (&row0)[NN],
                                                  int lane, int first, int step) {
  const int r16 = lane & 15, g8 = (lane >> 4) * 8;
#pragma unroll
  for (int j = 0; j < TT; ++j) {
    left[j] = left[j] < lo.n_ad ? left[j] : -1;
    half[j] = -1;
  }
  int round = 0;                               // an adapter's first
  for (;;) {
    int a = -1;
#pragma unroll
    for (int j = 0; j < TT; ++j) {
      const unsigned long long todo = __ballot(left[j] >= 0);
      if (a < 0 && todo) a = __builtin_amdgcn_readlane(left[j], __builtin_ctzll(todo));
    }
    if (a < 0) break;
    for (int c0 = 0; c0 < lo.r; c0 += 32) {
      if ((round + c0 / 32) % step != first) continue;           // uniform
#pragma unroll
      for (int j = 0; j < TT; ++j) half[j] = left[j] == a ? c0 / 32 : half[j];
    }
    for (int p = 0; p < lo.n_proj; ++p) {
      // projection p's, by masks: the compiler turns a choice into an address that depends on p, and `lo` would live in scratch memory
      const unsigned long long m0 = 0ull - (p == 0), m1 = 0ull - (p == 1), m2 = 0ull - (p == 2);
      const elt* Bp = (const elt*)(((uintptr_t)lo.B[0] & m0) | ((uintptr_t)lo.B[1] & m1) | ((uintptr_t)lo.B[2] & m2));
      const int begin = (lo.n_begin[0] & (int)m0) | (lo.n_begin[1] & (int)m1) | (lo.n_begin[2] & (int)m2);
      const int rows = (lo.n_rows[0] & (int)m0) | (lo.n_rows[1] & (int)m1) | (lo.n_rows[2] & (int)m2);
      bool has = false;
#pragma unroll
      for (int i = 0; i < NN; ++i) has = has || (row0[i] < begin + rows && row0[i] + 16 > begin);
      if (!has) continue;                      // uniform
      const float* vp = lo.v + (size_t)p * lo.ranges * T * lo.r;
      for (int c0 = 0; c0 < lo.r; c0 += 32) {
        if ((round + c0 / 32) % step != first) continue;         // uniform
        const int c = c0 + g8;                 // this lane's eight ranks (past r: zeros)
        eltx8 bf[NN];
#pragma unroll
        for (int i = 0; i < NN; ++i) {
          const int row = row0[i] + r16 - begin;
          bf[i] = c < lo.r && row >= 0 && row < rows ? ld8(Bp + ((size_t)a * rows + row) * lo.r + c) : eltx8{0, 0, 0, 0, 0, 0, 0, 0};
        }
#pragma unroll
        for (int j = 0; j < TT; ++j) {
          const int t = t0 + j * 16 + r16;
          const float* q = vp + (size_t)(t < T ? t : T - 1) * lo.r + (c < lo.r ? c : 0);
          f32x4 s0 = f32x4{0.f, 0.f, 0.f, 0.f}, s1 = s0;
          auto add_ranges = [&](int first) {
            f32x4 x0[DELTA_RANGES], x1[DELTA_RANGES];
#pragma unroll
            for (int s = 0; s < DELTA_RANGES; ++s) {             // (past the last range: that one again, not added)
              const float* qs = q + (size_t)(first + s < lo.ranges ? first + s : lo.ranges - 1) * T * lo.r;
              x0[s] = *reinterpret_cast<const f32x4*>(qs);
              x1[s] = *reinterpret_cast<const f32x4*>(qs + 4);
            }
#pragma unroll
            for (int s = 0; s < DELTA_RANGES; ++s) {
              s0 = first + s < lo.ranges ? s0 + x0[s] : s0;
              s1 = first + s < lo.ranges ? s1 + x1[s] : s1;
            }
          };
          add_ranges(0);
          if constexpr (V32) {
            if (lo.ranges > DELTA_RANGES) add_ranges(DELTA_RANGES);        // uniform
          }
          const bool of_a = left[j] == a && c < lo.r;            // (others': whatever lies there is replaced)
          float f[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) f[e] = of_a ? (e < 4 ? s0[e & 3] : s1[e & 3]) * lo.scaling : 0.f;
          eltx8 hi, low;
          Col32 col;
          if constexpr (V32) {
            col = col32_of(f);
          } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              hi[e] = (elt)f[e];
              low[e] = (elt)(f[e] - (float)hi[e]);
            }
          }
#pragma unroll
          for (int i = 0; i < NN; ++i) {
            f32x4 sum;
            if constexpr (V32) sum = mfma_16x16x32_col32(bf[i], col, acc[i][j]);
            else sum = mfma_16x16x32(bf[i], low, mfma_16x16x32(bf[i], hi, acc[i][j]));
            const bool of_p = row0[i] < begin + rows && row0[i] + 16 > begin;    // uniform
            acc[i][j] = left[j] == a && of_p ? sum : acc[i][j];
          }
        }
      }
    }
#pragma unroll
    for (int j = 0; j < TT; ++j) left[j] = left[j] == a ? -1 : left[j];
    round += (lo.r + 31) / 32;
  }
}
#endif
