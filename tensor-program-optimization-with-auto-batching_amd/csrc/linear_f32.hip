// Linear layers of the fp32 build:  y[T, N] (=|+=) alpha x[T, K] . W[N, K]^T  in IEEE fp32 on the matrix cores
// (v_mfma_f32_16x16x4_f32: products and sums in fp32), plain, per head (a batch of small matrices) or per expert (token tiles
// of a routing plan).
#include <type_traits>

#include "common.h"
#include "moe.h"

namespace {

constexpr int FB = 64;       // tokens of a block
constexpr int FW = 8;        // waves of a workgroup
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));   // 16 bytes at any element

struct F32Linear {
  float* y;
  const float* x;
  const float* W;
  long ldx, ldy;
  long hx, hy;               // head strides of x and y (blockIdx.z = head; the weights of a head are [N, K] blocks)
  int T, K, N;
  int tb;                    // tokens of a block (without a plan)
  float alpha;
  int accumulate, act;       // act: MLORA_ACT_*
  int gather, scatter, top;  // expert tiles (blockIdx.y = tile): gather: x row = entry / top; scatter: y row = entry
};

// The fp32 16 x 16 x 4 product takes one element per lane: a lane holds 4 consecutive k of its row, element e of the four
// k-groups of 16 lanes is one MFMA (any order of k serves, as long as both operands have the same).
//
// At T x K x N = 299 x 2048 x 2048: 42 us (60 TFLOP/s), 4 x 2048 x 11264: 20 us (4.6 TB/s), 4096 x 2048 x 11264: 1626 us
// (116 TFLOP/s).  The vector ALUs (64 x 64 blocks, both operands staged through LDS behind two barriers per 16 k): 122, 139 (one token),
// 2415 us.

// Adds the sums of the waves that share K, in their order, and stores.  red [KW][tiles][lane]: four rows n of a token; tile = row
// tile * RT + token tile.
template <int KW, int TILES, int RT>
__device__ __forceinline__ void f32_store(const F32Linear& a, const MoePlan& plan, int grouped, float* __restrict__ y, int n0, int t0, int t1,
                                          const f32x4* red) {
  for (int o = threadIdx.x; o < TILES * 64; o += FW * WAVE) {
    const int tile = o >> 6, l = o & 63;
    f32x4 v = red[o];
#pragma unroll
    for (int q = 1; q < KW; ++q) v += red[q * TILES * 64 + o];
    int t = t0 + tile % RT * 16 + (l & 15);
    const int n = n0 + tile / RT * 16 + (l >> 4) * 4;
    if (t >= t1 || n >= a.N) continue;
    if (grouped && a.scatter) t = plan.perm[t];
    float* p = y + t * a.ldy + n;
    v *= a.alpha;
    if (a.act == MLORA_ACT_RELU2) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        v[r] = fmaxf(v[r], 0.f);
        v[r] *= v[r];
      }
    }
    if (n + 4 <= a.N) {
      f32x4u* q = reinterpret_cast<f32x4u*>(p);
      *q = a.accumulate ? *q + v : v;
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (n + r < a.N) p[r] = a.accumulate ? p[r] + v[r] : v[r];
    }
  }
}

__device__ __forceinline__ f32x4 mfma_f32(const f32x4& w, const f32x4& x, f32x4 c) {
#pragma unroll
  for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(w[e], x[e], c, 0, 0, 0);
  return c;
}

// 16 weight rows per workgroup, up to 64 tokens (RT tiles of 16, as many as the block has): all eight waves share K, 32 k at a
// time in turn, so that together they read whole lines.  Operands go straight into registers, D stages ahead.  For few tokens
// or rows: bound by the stream of W and its latency; x is read again by every workgroup, through the first two cache levels.
template <int RT>
__device__ __forceinline__ void f32_thin(const F32Linear& a, const MoePlan& plan, int grouped, const float* __restrict__ x, const float* __restrict__ W,
                                         float* __restrict__ y, int n0, int t0, int t1, f32x4* red) {
  constexpr int D = RT == 1 ? 4 : RT <= 3 ? 3 : 2;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
  const float* wp = W + (size_t)(n0 + r16 < a.N ? n0 + r16 : a.N - 1) * a.K + g * 4;
  const float* xp[RT];
#pragma unroll
  for (int j = 0; j < RT; ++j) {
    int t = t0 + j * 16 + r16;
    t = t < t1 ? t : t1 - 1;
    if (grouped && a.gather) t = plan.perm[t] / a.top;
    xp[j] = x + t * a.ldx + g * 4;
  }
  f32x4 acc[RT], wf[D][2], xf[D][RT][2];
#pragma unroll
  for (int j = 0; j < RT; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int steps = (a.K + 31) / 32;              // of 32 k; the last one may have 16
  auto load = [&](auto S, int p) {
    constexpr int s = decltype(S)::value;
    const int k = (p < steps ? p : 0) * 32, k1 = k + 16 < a.K ? k + 16 : k;     // past the end: valid addresses, not multiplied
    wf[s][0] = *reinterpret_cast<const f32x4u*>(wp + k);
    wf[s][1] = *reinterpret_cast<const f32x4u*>(wp + k1);
#pragma unroll
    for (int j = 0; j < RT; ++j) {
      xf[s][j][0] = *reinterpret_cast<const f32x4u*>(xp[j] + k);
      xf[s][j][1] = *reinterpret_cast<const f32x4u*>(xp[j] + k1);
    }
  };
  auto turn = [&](auto S, int p) {
    constexpr int s = decltype(S)::value;
    load(std::integral_constant<int, (s + D - 1) % D>(), p + (D - 1) * FW);
    if (p >= steps) return;                       // uniform
#pragma unroll
    for (int j = 0; j < RT; ++j) acc[j] = mfma_f32(wf[s][0], xf[s][j][0], acc[j]);
    if (p * 32 + 16 < a.K) {
#pragma unroll
      for (int j = 0; j < RT; ++j) acc[j] = mfma_f32(wf[s][1], xf[s][j][1], acc[j]);
    }
  };
  load(std::integral_constant<int, 0>(), wave);
  if constexpr (D > 2) load(std::integral_constant<int, 1>(), wave + FW);
  if constexpr (D > 3) load(std::integral_constant<int, 2>(), wave + 2 * FW);
  for (int p = wave; p < steps; p += D * FW) {
    turn(std::integral_constant<int, 0>(), p);
    turn(std::integral_constant<int, 1>(), p + FW);
    if constexpr (D > 2) turn(std::integral_constant<int, 2>(), p + 2 * FW);
    if constexpr (D > 3) turn(std::integral_constant<int, 3>(), p + 3 * FW);
  }
#pragma unroll
  for (int j = 0; j < RT; ++j) red[(wave * RT + j) * 64 + lane] = acc[j];
  __syncthreads();
  f32_store<FW, RT, RT>(a, plan, grouped, y, n0, t0, t1, red);
}

// FN * 16 weight rows by up to 64 tokens: four waves share the rows (FN / 4 tiles each, all tokens), twice, for the two halves
// of every 64 k.  Both operands go from global memory straight into an LDS ring that is NST - 1 stages of 64 k ahead, one bare barrier per stage.  Bound by the matrix cores (157 TFLOP/s nominal) or, for few
// tokens, by what a workgroup takes in.  NST: a deep ring where a workgroup has a compute unit to itself, one of two stages where two
// share it and their waits overlap.  DIRECT: operands are 16-byte aligned; others go through registers.  SUMS: of a wave for an output.  Four, by
// element e, make eight with the two halves of K, as many as f32_thin has: the rounding of a sum does not depend on which form a size takes
// (4 x 2048 x 11264, error against 64 bits 2.9e-7 here and there, 5.7e-7 with one).  They cost registers, not time (20.3 us both), but where
// four workgroups share a compute unit: one, for a K of one stage (4000 x 64 x 4096 32 us, with four 39), which f32_thin adds in two chains as well.
template <int FN, int RT, int NST, bool DIRECT, int SUMS>
__device__ __forceinline__ void f32_wide(const F32Linear& a, const MoePlan& plan, int grouped, const float* __restrict__ x, const float* __restrict__ W,
                                         float* __restrict__ y, int n0, int t0, int t1, f32x4* smem) {
  constexpr int RW = FN / 4, SF = FN + RT, LF = 4 * SF, LQ = (LF + FW - 1) / FW;   // row tiles of a stage, requests for it (four rows x 64 k), of a wave
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
  // request f = wave + 8 q of a stage: four rows of weight tile or (behind those) token tile f / 4, 64 k each: whole lines.  (16 rows of 16 k a
  // request, as the lanes multiply them, are half lines: 16 x 2048 x 11264 25 -> 18 us, 299 x 5632 x 2048 125 -> 109, 192 entries over 64 experts of 2048 x
  // 1408 134 -> 121.)  A row's quad c lies in LDS at place c ^ row, so that 16 rows' quads fall on different banks.
  const float* src[LQ];
  int fd[LQ], fk[LQ];
#pragma unroll
  for (int q = 0; q < LQ; ++q) {
    int f = wave + FW * q;
    f = f < LF ? f : LF - 1;                      // (twice the same: every wave has LQ requests per stage)
    fd[q] = f;
    const int row = (f & 3) * 4 + g;
    f >>= 2;
    fk[q] = (r16 ^ row) * 4;
    if (f < FN) {
      const int n = n0 + f * 16 + row;
      src[q] = W + (size_t)(n < a.N ? n : a.N - 1) * a.K;
    } else {
      int t = t0 + (f - FN) * 16 + row;
      t = t < t1 ? t : t1 - 1;
      if (grouped && a.gather) t = plan.perm[t] / a.top;
      src[q] = x + t * a.ldx;
    }
  }
  const int nst = (a.K + 63) / 64;
  int slot = 0;                                   // of the stage requested next
  auto request = [&](int s) {
#pragma unroll
    for (int q = 0; q < LQ; ++q) {
      const float* p = src[q] + (s * 64 + fk[q] < a.K ? s * 64 + fk[q] : 0);      // past the end: a valid address, not multiplied
      f32x4* d = smem + (slot * LF + fd[q]) * 64;
      if constexpr (DIRECT)
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)p, (__attribute__((address_space(3))) void*)d, 16, 0, 0);
      else
        d[lane] = *reinterpret_cast<const f32x4u*>(p);
    }
    slot = slot + 1 < NST ? slot + 1 : 0;
  };
  const int rg = wave & 3, kh = wave >> 2;
  f32x4 acc[RW][RT][SUMS];
#pragma unroll
  for (int i = 0; i < RW; ++i)
#pragma unroll
    for (int j = 0; j < RT; ++j)
#pragma unroll
      for (int e = 0; e < SUMS; ++e) acc[i][j][e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < NST - 1; ++s) request(s);
  int rd = 0;
  for (int s = 0; s < nst; ++s) {
    // stage s has landed (this wave's share: at most the NST - 2 stages behind it in flight; everybody's: the barrier), and
    // everybody is done with the slot of stage s - 1, which is requested anew
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((NST - 2) * LQ) : "memory");
    bare_barrier();
    if (NST > 2 || s + 1 < nst) request(s + NST - 1);       // (the wait counts the requests past the end of a deeper ring)
    const f32x4* st = smem + rd * LF * 64 + r16 * 16;
    rd = rd + 1 < NST ? rd + 1 : 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (s * 64 + kh * 32 + h * 16 >= a.K) break;                   // uniform
      const int at = (kh * 8 + h * 4 + g) ^ r16;
      f32x4 w[RW], xv[RT];
#pragma unroll
      for (int i = 0; i < RW; ++i) w[i] = st[(rg * RW + i) * 256 + at];
#pragma unroll
      for (int j = 0; j < RT; ++j) xv[j] = st[(FN + j) * 256 + at];
#pragma unroll
      for (int i = 0; i < RW; ++i)
#pragma unroll
        for (int j = 0; j < RT; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][j][e % SUMS] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[i][e], xv[j][e], acc[i][j][e % SUMS], 0, 0, 0);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                   // the requests past the end, too: the ring becomes the waves' sums
  __syncthreads();
#pragma unroll
  for (int i = 0; i < RW; ++i)
#pragma unroll
    for (int j = 0; j < RT; ++j) {
      f32x4 v = acc[i][j][0];
#pragma unroll
      for (int e = 1; e < SUMS; ++e) v += acc[i][j][e];
      smem[((kh * 4 + rg) * RW * RT + i * RT + j) * 64 + lane] = v;
    }
  __syncthreads();
  f32_store<2, FN * RT, RT>(a, plan, grouped, y, n0, t0, t1, smem);
}

// FN: row tiles of a workgroup (1: f32_thin)
template <int FN, int NST, bool DIRECT, int SUMS>
__global__ __launch_bounds__(FW* WAVE, 2) void linear_f32_kernel(F32Linear a, MoePlan plan, int grouped) {
  extern __shared__ __align__(16) f32x4 f32_smem[];
  const int n0 = blockIdx.x * FN * 16;
  int t0 = blockIdx.y * a.tb, t1 = a.T;
  const float* W = a.W + (size_t)blockIdx.z * a.N * a.K;
  const float* x = a.x + blockIdx.z * a.hx;
  float* y = a.y + blockIdx.z * a.hy;
  if (grouped) {
    if ((int)blockIdx.y >= *plan.n_tiles) return;
    const int4 tile = plan.tiles[blockIdx.y];
    W = a.W + (size_t)tile.x * a.N * a.K;
    t0 = tile.y;
    t1 = tile.y + tile.z;
  }
  t1 = t1 < t0 + a.tb ? t1 : t0 + a.tb;
  const int rt = __builtin_amdgcn_readfirstlane((t1 - t0 + 15) >> 4);
  auto block = [&](auto RT) {
    if constexpr (FN == 1) f32_thin<decltype(RT)::value>(a, plan, grouped, x, W, y, n0, t0, t1, f32_smem);
    else f32_wide<FN, decltype(RT)::value, NST, DIRECT, SUMS>(a, plan, grouped, x, W, y, n0, t0, t1, f32_smem);
  };
  if (rt == 1) block(std::integral_constant<int, 1>());
  else if (rt == 2) block(std::integral_constant<int, 2>());
  else if (rt == 3) block(std::integral_constant<int, 3>());
  else block(std::integral_constant<int, 4>());
}

int f32_n_cu() {
  static const int n_cu = [] {
    int dev = 0, cu = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cu <= 0) cu = 256;
    return cu;
  }();
  return n_cu;
}

template <int FN, int NST = 0, bool DIRECT = true, int SUMS = 4>
int launch_f32(const char* who, const F32Linear& a, const MoePlan& plan, int grouped, int row_blocks, int heads, hipStream_t stream) {
  constexpr size_t stage = 4 * (FN + 4) * 1024, most = FN == 1 ? FW * 4 * 1024 : NST * stage;      // the waves' sums, or the ring (which these fit)
  const size_t lds = SUMS == 1 ? stage : most;    // (a K of one stage)
  static const hipError_t configured =               // the attribute is per kernel, set once per process, by one thread
      hipFuncSetAttribute((const void*)linear_f32_kernel<FN, NST, DIRECT, SUMS>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)most);
  if (configured != hipSuccess) return mlora_set_error(MLORA_ERR_LAUNCH, "%s: cannot reserve %zu bytes of LDS: %s", who, lds, hipGetErrorString(configured));
  hipLaunchKernelGGL((linear_f32_kernel<FN, NST, DIRECT, SUMS>), dim3(ceil_div(a.N, FN * 16), row_blocks, heads), dim3(FW * WAVE), lds, stream, a, plan, grouped);
  return mlora_launch_status(who);
}

// FN row tiles of 16 and tb tokens of a workgroup's block; a ring of NST stages, SUMS sums of a wave for an output (f32_wide)
struct F32Form {
  int fn, tb, nst, sums;
};

F32Form choose(int T, int K, int N, bool grouped, int row_blocks, int heads) {
  // The form that finishes first, m token tiles of 16 and k times 2048 k: rounds of the compute units times what a workgroup takes, in us but for what a
  // launch costs in any form.  16 rows: 5.6 + (3 + 2.2 m) k, and at least 6 ns per k of the first 256, one stage of every wave; without a plan its token
  // blocks are of 16, 32 or 64, as leaves least.  64 rows, ring of four: (2.5 + 10.9 m) k, at least 17.2 k, and 2.2; ring of two: (4.4 + 9.9 m) k two
  // together, (1.1 + 9.1 m) k, at least 26.5 k, alone in the last round, and 0.94 of waiting, which four share where K is one stage.  128 rows: (5.7 +
  // 8.9 m) k, at least 19.6 k, and 3.  Fitted to the choices over 882 sizes of 1 to 4096 tokens, K of 16 to 11008, 16 to 36000 rows, heads and experts' plans, weights from
  // memory: the choice takes 1.1 % longer than the best form on average, 40 % at most (12 entries over 16 experts of 1408 x 2048 31 us instead of 22; 219 x 48 x 224 3.8 instead of 2.9).  Costs fitted to
  // K from 512 on took 2.5 % longer: 247 x 2864 x 4384 and 500 x 256 x 304 went to 16 rows.  Tokens x K x rows, 16 rows in blocks of 16 tokens / 64
  // tokens / 64 rows with four stages / with two / 128, us: 1 x 2048 x 2048 9 / 9 / 17 / 20 / 29, 4 x 2048 x 11264 24 / 25 / 19 / 29 / 30, 32 x 2048 x 2048 12 / 17 /
  // 25 / 25 / 43, 299 x 2048 x 128 12 / 22 / 41 / 41 / 74, 299 x 2048 x 2048 97 / 63 / 43 / 44 / 76, 24 x 2048 x 32000 141 / 108 / 55 / 52 / 48, 299 x 2048 x 11264
  // 495 / 269 / 156 / 154 / 149, 500 x 256 x 304 20 / 8.9 / 8.3 / 7.8 / 13, 247 x 2864 x 4384 167 / 132 / 114 / 110 / 107.  Over a plan: its tiles as far as the host can tell,
  // half of the experts' last ones.
  const int full = T / FB, experts = row_blocks - full, tiles = !grouped ? row_blocks : full + experts / 2 > experts ? full + experts / 2 : experts;
  const double m = (double)(grouped ? T / tiles : T < FB ? T : FB) / 16, k = K / 2048.0;
  const long cu = f32_n_cu(), col = (long)tiles * heads, n4 = ceil_div(N, 64) * col, n8 = ceil_div(N, 128) * col;
  auto rounds = [](long blocks, long slots) { return (double)((blocks + slots - 1) / slots); };
  auto thin = [&](long col, double m) {
    const long n1 = ceil_div(N, 16) * col;
    const double r1 = m > 0.5 || n1 < cu ? rounds(n1, cu) : (double)n1 / cu;     // (few tokens: the next workgroups start as units are free)
    return r1 * fmax(0.006 * (K < 256 ? K : 256), 5.6 + (3 + 2.2 * m) * k);
  };
  int tb = FB;
  double c1 = thin(col, m);
  for (int t = FB / 2; !grouped && t >= 16 && ceil_div(T, t) <= 65535; t /= 2) {
    if (t >= T) continue;                          // one block either way
    const double c = thin((long)ceil_div(T, t) * heads, t / 16.0);
    if (c < c1) {
      c1 = c;
      tb = t;
    }
  }
  const double c4 = rounds(n4, cu) * (fmax(17.2, 2.5 + 10.9 * m) * k + 2.2);
  const int alone = n4 % (2 * cu) > 0 && n4 % (2 * cu) <= cu ? 1 : 0;
  const double c2 = ((rounds(n4, 2 * cu) - alone) * (4.4 + 9.9 * m) + alone * fmax(26.5, 1.1 + 9.1 * m)) * k + rounds(n4, (K <= 64 ? 4 : 2) * cu) * 0.94;
  const double c8 = rounds(n8, cu) * (fmax(19.6, 5.7 + 8.9 * m) * k + 3);
  if (c1 <= c4 && c1 <= c2 && c1 <= c8) return {1, tb, 0, 4};
  if (c8 < c4 && c8 < c2) return {8, FB, 3, 4};
  if (c4 < c2) return {4, FB, 4, 4};
  return {4, FB, 2, K <= 64 ? 1 : 4};
}

int launch(const char* who, F32Linear a, const MoePlan& plan, int grouped, int row_blocks, int heads, void* stream) {
  MLORA_CHECK(a.K % 16 == 0 && a.ldx % 4 == 0 && a.hx % 4 == 0 && row_blocks <= 65535 && heads <= 65535, MLORA_ERR_UNSUPPORTED,
              "%s: need K %% 16 == 0 and rows aligned to 16 bytes (T=%d K=%d N=%d)", who, a.T, a.K, a.N);
  const F32Form f = choose(a.T, a.K, a.N, grouped, row_blocks, heads);
  const bool direct = (((uintptr_t)a.x | (uintptr_t)a.W) & 15) == 0;           // x may begin at any column of a wider tensor
  const hipStream_t s = (hipStream_t)stream;
  a.tb = f.tb;
  if (f.fn == 1) return launch_f32<1>(who, a, plan, grouped, grouped ? row_blocks : ceil_div(a.T, a.tb), heads, s);
  if (!direct && f.sums == 1) return launch_f32<4, 2, false, 1>(who, a, plan, grouped, row_blocks, heads, s);   // (the bits of aligned operands)
  if (!direct) return launch_f32<4, 2, false>(who, a, plan, grouped, row_blocks, heads, s);
  if (f.fn == 8) return launch_f32<8, 3>(who, a, plan, grouped, row_blocks, heads, s);
  if (f.nst == 4) return launch_f32<4, 4>(who, a, plan, grouped, row_blocks, heads, s);
  if (f.sums == 1) return launch_f32<4, 2, true, 1>(who, a, plan, grouped, row_blocks, heads, s);
  return launch_f32<4, 2>(who, a, plan, grouped, row_blocks, heads, s);
}

}  // namespace

// how mlora_linear takes a size: weight rows of a workgroup, its tokens and the stages of its ring, a byte each
extern "C" int mlora_linear_block(int T, int K, int N) {
  const F32Form f = choose(T, K, N, false, ceil_div(T, FB), 1);
  return f.fn << 20 | f.tb << 8 | f.nst;
}

extern "C" int mlora_linear(void* y, int y_dtype, int mode, const void* x, int ldx, const void* W, int T, int K, int N, void* stream) {
  MLORA_CHECK(y && x && W && T >= 0 && K > 0 && N > 0 && ldx >= K, MLORA_ERR_INVALID, "linear: null pointer or bad shape T=%d K=%d N=%d", T, K, N);
  if (T == 0) return MLORA_OK;
  F32Linear a = {};
  a.y = (float*)y; a.x = (const float*)x; a.W = (const float*)W;
  a.ldx = ldx; a.ldy = N; a.T = T; a.K = K; a.N = N; a.alpha = 1.f; a.accumulate = mode == MLORA_ACCUMULATE;
  return launch("linear", a, MoePlan(), 0, ceil_div(T, FB), 1, stream);
}

extern "C" int mlora_head_linear(void* y, int y_layout, long ldy, long head_y, const void* x, long ldx, long head_x, const void* W, int heads, int T,
                                 int K, int N, float alpha, void* stream) {
  MLORA_CHECK(y && x && W && T >= 0 && K > 0 && N > 0 && heads > 0, MLORA_ERR_INVALID, "head_linear: null pointer or bad shape");
  MLORA_CHECK(y_layout == MLORA_ROWMAJOR, MLORA_ERR_UNSUPPORTED, "head_linear: fragment order is for 16-bit elements");
  if (T == 0) return MLORA_OK;
  F32Linear a = {};
  a.y = (float*)y; a.x = (const float*)x; a.W = (const float*)W;
  a.ldx = ldx; a.ldy = ldy; a.hx = head_x; a.hy = head_y; a.T = T; a.K = K; a.N = N; a.alpha = alpha;
  return launch("head_linear", a, MoePlan(), 0, ceil_div(T, FB), heads, stream);
}

extern "C" int mlora_moe_linear(void* y, const void* x, const void* W, const int32_t* perm, const int32_t* tiles, const int32_t* n_tiles,
                                int tile_rows, int max_tiles, int places, int T, int K, int N, int top, int stage, int act, float alpha,
                                void* workspace, size_t workspace_elems, void* stream) {
  MLORA_CHECK(y && x && W && perm && tiles && n_tiles && T >= 0 && K > 0 && N > 0 && top > 0 && tile_rows == FB && max_tiles >= 0, MLORA_ERR_INVALID,
              "moe_linear: null pointer or bad shape (tile_rows=%d tiles=%d)", tile_rows, max_tiles);
  (void)places; (void)workspace; (void)workspace_elems;      // the matrix-core form's
  if (T == 0 || max_tiles == 0) return MLORA_OK;
  F32Linear a = {};
  a.y = (float*)y; a.x = (const float*)x; a.W = (const float*)W;
  a.ldx = K; a.ldy = N; a.T = T * top; a.K = K; a.N = N; a.alpha = alpha; a.act = act; a.top = top;
  a.gather = stage == MLORA_MOE_UP;
  a.scatter = stage == MLORA_MOE_DOWN;
  MoePlan p;
  p.perm = perm; p.tiles = (const int4*)tiles; p.n_tiles = n_tiles;
  return launch("moe_linear", a, p, 1, max_tiles, 1, stream);
}
