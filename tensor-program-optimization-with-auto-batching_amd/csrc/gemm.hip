// Prefill-time base linear for gfx950:  y[T, N] (=|+=) x[T, K] . W[N, K]^T  for any T (MFMA-bound).
//
// Three kernels, by operand layout and problem size:
//   gemm_kernel      row-major or fragment-ordered W, fragments loaded straight from global memory into registers
//                    (both operands are K-contiguous, which is what v_mfma_f32_16x16x32_f16 wants: a lane holds 8
//                    consecutive k of one row); a wave owns 64 x 64 outputs.  Any shape; the small-T workhorse.
//   gemm_lds_kernel  fragment-ordered W, register-staged LDS double buffer; 256 x 64 or 256 x 256 blocks.
//   gemm_pp_kernel   fragment-ordered W and row-major or fragment-ordered x, both copied from global memory straight
//                    into a four-stage LDS ring; persistent 256 x 256 blocks, eight waves.  The large-T kernel.
// All three add the 32-k MFMA steps of an output in ascending k into one accumulator, so their results are the same
// bits.
#include <type_traits>

#include "lora_device.h"
#include "moe.h"

int mlora_check_linear(const char* who, const void* y, int y_dtype, int mode, const void* x, int ldx, const void* W,
                       int T, int K, int N);

namespace {

enum { OUT_F16 = 0, OUT_F32 = 1, OUT_ACC_F32 = 2, OUT_SILU = 3, OUT_CLIP = 4, OUT_RELU2 = 5 };   // OUT_SILU, OUT_CLIP: a gated product (MLORA_GLU_*), OUT_RELU2: max(alpha y, 0)^2, all in fragment order

// compute units of the current device (0 if it cannot be asked), read once
int gemm_n_cu() {
  static const int n_cu = [] {
    int dev = 0, cu = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) cu = 0;
    return cu;
  }();
  return n_cu;
}

constexpr int WT = 4;   // 16-wide MFMA tiles per wave along N and along T

template <int OUT, bool PACKED>
__global__ __launch_bounds__(256) void gemm_kernel(void* __restrict__ yv, const elt* __restrict__ x, int ldx,
                                                   const elt* __restrict__ W, int T, int K, int N) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r16 = lane & 15, kg = lane >> 4;
  const int n0 = blockIdx.x * 128 + (wave & 1) * 64;
  const int t0 = blockIdx.y * 128 + (wave >> 1) * 64;
  if (n0 >= N || t0 >= T) return;

  constexpr int WSTEP = PACKED ? 512 : 32;   // elements between consecutive k-steps of one fragment stream
  const int tiles = (N + 15) / 16;
  const elt* wp[WT];
  const elt* xp[WT];
#pragma unroll
  for (int i = 0; i < WT; ++i) {
    if constexpr (PACKED) {
      int nt = n0 / 16 + i;
      nt = nt < tiles ? nt : tiles - 1;
      wp[i] = W + ((size_t)nt * (K / 32)) * 512 + lane * 8;
    } else {
      int n = n0 + i * 16 + r16;
      n = n < N ? n : N - 1;
      wp[i] = W + (size_t)n * K + kg * 8;
    }
    int t = t0 + i * 16 + r16;
    t = t < T ? t : T - 1;
    xp[i] = x + (size_t)t * ldx + kg * 8;
  }
  f32x4 acc[WT][WT];
#pragma unroll
  for (int i = 0; i < WT; ++i)
#pragma unroll
    for (int j = 0; j < WT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  eltx8 a[WT], b[WT];
#pragma unroll
  for (int i = 0; i < WT; ++i) {
    a[i] = ld8(wp[i]);
    b[i] = ld8(xp[i]);
  }
  const int KB = K / 32;
  for (int ks = 1; ks <= KB; ++ks) {
    eltx8 an[WT], bn[WT];
    const int kc = ks < KB ? ks : 0;   // the last prefetch wraps to a valid address and is discarded
#pragma unroll
    for (int i = 0; i < WT; ++i) {
      an[i] = ld8(wp[i] + (size_t)kc * WSTEP);
      bn[i] = ld8(xp[i] + kc * 32);
    }
#pragma unroll
    for (int i = 0; i < WT; ++i)
#pragma unroll
      for (int j = 0; j < WT; ++j) acc[i][j] = mfma_16x16x32(a[i], b[j], acc[i][j]);
#pragma unroll
    for (int i = 0; i < WT; ++i) {
      a[i] = an[i];
      b[i] = bn[i];
    }
  }

  const int g = lane >> 4;
#pragma unroll
  for (int j = 0; j < WT; ++j) {
    const int t = t0 + j * 16 + r16;
    if (t >= T) continue;
#pragma unroll
    for (int i = 0; i < WT; ++i) {
      const int n = n0 + i * 16 + g * 4;
      if (n >= N) continue;
      const size_t o = (size_t)t * N + n;
      const f32x4 s = acc[i][j];
      if constexpr (OUT == OUT_F16) {
        *reinterpret_cast<eltx4*>((elt*)yv + o) = eltx4{(elt)s[0], (elt)s[1], (elt)s[2], (elt)s[3]};
      } else if constexpr (OUT == OUT_F32) {
        *reinterpret_cast<f32x4*>((float*)yv + o) = s;
      } else {
        f32x4* p = reinterpret_cast<f32x4*>((float*)yv + o);
        *p = *p + s;
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
// LDS-staged variant for fragment-ordered weights.  In its large shape a workgroup of 4 waves owns a 256-token x
// 256-column output block, a wave 128 x 128 of it (8 x 8 MFMA tiles; the 256 accumulator registers live in the
// accumulation half of the register file at one wave per SIMD).  A stage is 64 k of both operands (2 x 32 KiB) staged through LDS in
// fragment order, double buffered: while the matrix cores work on one buffer, the next stage's global loads are in
// flight and are written to the other buffer, one barrier per stage.  Weight fragments are copied as they lie in
// memory (contiguous 1 KiB); the token rows are read 64 contiguous bytes at a time and transposed into fragment
// order by the LDS write (with an XOR on the token slot that keeps every quarter-wave write conflict-free).
// Per stage and CU: 64 KiB from L2 for 2 x 64 x 4 MFMAs (2048 MFMA cycles per SIMD): 32 B/clk, half the L1 rate;
// LDS traffic 64 KiB written + 128 KiB read.
// ---------------------------------------------------------------------------------------------
constexpr int LBK = 64;              // k per stage

// FT x FN: 16-row fragments of tokens / of weight rows per block; WT x WN: MFMA tiles of a wave (FT/WT * FN/WN == 4 waves)
template <int OUT, int FT, int FN, int WT_, int WN_>
__global__ __launch_bounds__(256) void gemm_lds_kernel(void* __restrict__ yv, const elt* __restrict__ x, int ldx,
                                                       const elt* __restrict__ Wp, int T, int K, int N) {
  static_assert((FT / WT_) * (FN / WN_) == 4, "four waves cover the block");
  constexpr int KS = LBK / 32;                      // 32-k steps per stage
  constexpr int WELEMS = KS * FN * 512, XELEMS = KS * FT * 512;   // fp16 elements of a stage: W, then x
  constexpr int STAGE = WELEMS + XELEMS;
  constexpr int WCH = KS * FN * WAVE / 256, XCH = KS * FT * WAVE / 256;   // 16-byte chunks per thread and stage
  static_assert(WCH >= 1 && XCH >= 1, "a stage gives every thread at least one chunk of each operand");
  extern __shared__ __align__(16) elt smem[];       // [2][STAGE]
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int n0 = blockIdx.x * FN * 16, t0 = blockIdx.y * FT * 16;
  constexpr int WAVES_N = FN / WN_;
  const int wn = wave % WAVES_N, wt = wave / WAVES_N;
  const int KB = K / 32;
  const int tiles = (N + 15) / 16;

  // chunk c = threadIdx.x + 256 j of an operand's stage: fragment f = c / 64 = ks * F + tile, lane slot l = c % 64
  const elt* wsrc[WCH];
  const elt* xsrc[XCH];
#pragma unroll
  for (int j = 0; j < WCH; ++j) {
    const int c = threadIdx.x + 256 * j;
    const int f = c >> 6, l = c & 63;
    const int ks = f / FN, tile = f % FN;
    int nt = n0 / 16 + tile;
    nt = nt < tiles ? nt : tiles - 1;               // columns past N: a valid fragment, results dropped
    wsrc[j] = Wp + ((size_t)nt * KB + ks) * 512 + l * 8;
  }
  // x chunks: 4 consecutive lanes read the 64 contiguous bytes (one 32-k step) of one token row, so a quarter-wave
  // covers 4 rows x 4 lane groups g.  The LDS slot of a token inside its 16-token fragment is XORed with 4 g: the 16
  // lanes of a quarter-wave then write 16 different slots (no bank conflict), and a read of a fragment stays a
  // permutation inside each 16-lane group.
  int xdst[XCH];
#pragma unroll
  for (int j = 0; j < XCH; ++j) {
    const int c2 = threadIdx.x + 256 * j;
    const int ks = c2 / (FT * 64), c = c2 % (FT * 64);
    const int row = c >> 2, gq = c & 3;
    int t = t0 + row;
    t = t < T ? t : T - 1;
    xsrc[j] = x + (size_t)t * ldx + ks * 32 + gq * 8;
    xdst[j] = ((ks * FT + (row >> 4)) * 64 + gq * 16 + ((row & 15) ^ (gq << 2))) * 8;
  }
  eltx8 wst[WCH], xst[XCH];
  auto load_stage = [&](int s) {                    // s: stage index; k-steps KS*s .. (the last may be past K)
#pragma unroll
    for (int j = 0; j < WCH; ++j) {
      const int ks = (threadIdx.x + 256 * j) / (64 * FN);
      const int kb = s * KS + ks;
      const int kc = kb < KB ? kb : KB - 1;         // past K: a valid address; that step is not multiplied
      wst[j] = ld8(wsrc[j] + (size_t)(kc - ks) * 512);
    }
#pragma unroll
    for (int j = 0; j < XCH; ++j) {
      const int ks = (threadIdx.x + 256 * j) / (FT * 64);
      const int kb = s * KS + ks;
      const int kc = kb < KB ? kb : KB - 1;
      xst[j] = ld8(xsrc[j] + (kc - ks) * 32);
    }
  };
  auto store_stage = [&](int buf) {
    elt* dst = smem + buf * STAGE;
#pragma unroll
    for (int j = 0; j < WCH; ++j) st8(dst + (threadIdx.x + 256 * j) * 8, wst[j]);
#pragma unroll
    for (int j = 0; j < XCH; ++j) st8(dst + WELEMS + xdst[j], xst[j]);
  };

  f32x4 acc[WN_][WT_];
#pragma unroll
  for (int i = 0; i < WN_; ++i)
#pragma unroll
    for (int j = 0; j < WT_; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int xslot = (lane & 48) + ((lane & 15) ^ ((lane >> 4) << 2));   // lane's token slot after the write-side XOR
  const int S = (KB + KS - 1) / KS;
  load_stage(0);
  store_stage(0);
  __syncthreads();
  for (int s = 0; s < S; ++s) {
    if (s + 1 < S) load_stage(s + 1);
    const elt* ws = smem + (s & 1) * STAGE;
    const elt* xs = ws + WELEMS;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if (s * KS + ks < KB) {                        // workgroup-uniform
        eltx8 a[WN_], b[WT_];
#pragma unroll
        for (int i = 0; i < WN_; ++i) a[i] = ld8(ws + (ks * FN + wn * WN_ + i) * 512 + lane * 8);
#pragma unroll
        for (int j = 0; j < WT_; ++j) b[j] = ld8(xs + (ks * FT + wt * WT_ + j) * 512 + xslot * 8);
#pragma unroll
        for (int i = 0; i < WN_; ++i)
#pragma unroll
          for (int j = 0; j < WT_; ++j) acc[i][j] = mfma_16x16x32(a[i], b[j], acc[i][j]);
      }
    }
    if (s + 1 < S) store_stage((s + 1) & 1);
    __syncthreads();
  }

  const int r16 = lane & 15, g = lane >> 4;
#pragma unroll
  for (int j = 0; j < WT_; ++j) {
    const int t = t0 + (wt * WT_ + j) * 16 + r16;
    if (t >= T) continue;
#pragma unroll
    for (int i = 0; i < WN_; ++i) {
      const int n = n0 + (wn * WN_ + i) * 16 + g * 4;
      if (n >= N) continue;
      const size_t o = (size_t)t * N + n;
      const f32x4 sacc = acc[i][j];
      if constexpr (OUT == OUT_F16) {
        *reinterpret_cast<eltx4*>((elt*)yv + o) = eltx4{(elt)sacc[0], (elt)sacc[1], (elt)sacc[2], (elt)sacc[3]};
      } else if constexpr (OUT == OUT_F32) {
        *reinterpret_cast<f32x4*>((float*)yv + o) = sacc;
      } else {
        f32x4* p = reinterpret_cast<f32x4*>((float*)yv + o);
        *p = *p + sacc;
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
// Eight-wave persistent variant for large token counts.  A workgroup owns 256 tokens x 256 weight rows at a time, a
// wave 64 tokens x 128 rows of it (4 x 8 MFMA tiles, 128 accumulator registers), two waves per SIMD, one workgroup
// per compute unit, which walks through its share of the output blocks.
//   * Both operands go from global memory straight into LDS (global_load_lds_dwordx4: no register staging, no LDS
//     store instructions) in fragment order, through a ring of four 32-k stages with three stages in flight ahead of
//     the one being multiplied.  A weight fragment is copied as it lies in memory.  A token fragment likewise when the
//     activations come in fragment order (x_tt > 0: Xf[k/32][t/16][4][16][8], one contiguous 1 KiB block per
//     fragment); from row-major activations it is gathered 16 rows x 64 bytes by the load's per-lane addresses - half
//     cache lines, which costs the load path a third of its speed.
//   * The ring runs on across block boundaries: while the last stages of a block are multiplied and its results are
//     stored, the first stages of the workgroup's next block are already in flight.
//   * The two waves of a SIMD take turns: half a stage apart, one multiplies (32 products, 512 cycles) while the other reads its
//     fragments from LDS, requests its share of a later stage and waits; a bare barrier, twice per stage, swaps them.  With all eight
//     waves in step behind one barrier per stage, reads of the next stage ahead of the products of this one, the matrix cores
//     were busy half of the time (0.52 of the cycles at 2.17 GHz, 4096 tokens x 12288 x 4096; now 0.72 at 1.85 GHz, where the
//     power limit begins).  bf16, then and now, us: 4096 x 12288 x 4096 319 -> 287, 4096 x 4096 x 4096 103 -> 94,
//     4096 x 22016 x 4096 614 -> 517, 8192 x 8192 x 8192 845 -> 696 (1.58 PFLOP/s).
//   * fp16 results cross a small LDS buffer so that a store instruction writes whole 128-byte lines of a token row.
// Blocks are numbered so that an XCD (workgroup id mod 8) works through a contiguous range of them, in bands of a few token
// blocks that share their weights and tokens in its L2 (block_of).
// ---------------------------------------------------------------------------------------------
constexpr int PP_WAVES = 8;
constexpr int PP_STAGES = 4;
constexpr int PP_F = 16;                       // 16-row fragments per block side (256 tokens, 256 weight rows)
constexpr int PP_STAGE_ELEMS = 2 * PP_F * 512; // fp16 elements of one 32-k stage: 16 weight fragments, then 16 token fragments
constexpr int PP_OUT_LD = 64 + 4;              // fp16 elements per token row of a wave's output staging (padded: conflict-free writes)
constexpr int PP_OUT_ELEMS = 16 * PP_OUT_LD;   // per wave: 16 tokens x 64 columns

// LoRA deltas that ride in the GEMM as extra k-steps: y = [x | v_hi | v_lo] . [W | B[a] | B[a]]^T for a 256-token block
// whose tokens all name adapter a (blk_adapter[block] >= 0), v = scaling * x . A[a]^T as fp16 hi + lo halves [T][r].
// Projections are row ranges of the fused weight, each with its own B table [n_ad][rows][r] (row-major, r in {32, 64})
// and its own v; a 256-row block lies inside one range (checked by the launcher).  n_proj == 0: a plain GEMM.
struct PPLora {
  const elt* B[3];
  const elt* vh[3];
  const elt* vl[3];
  int n_begin[3], n_rows[3];
  int n_proj, r;
  const int32_t* blk_adapter;
};

// A grouped GEMM over a routing plan (moe.h): a token block is a tile of the plan - up to 256 places of one expert, whose
// weights it is multiplied with.  Places are in fragment order (x_tt tiles of 16).  Results go to fragment-ordered places
// (OUT_RELU2) or, row-major, to the entries the places stand for (OUT_F16), times alpha.
struct PPGroup {
  MoePlan plan;
  size_t w_elems;
  float alpha;
};
// With OUT_SILU the group's up stage ends in a gated product: an expert's weights are its gate rows, then its up rows.

typedef int i32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ unsigned long long uniform64(unsigned long long v) {
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v), hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
  return ((unsigned long long)hi << 32) | lo;
}

// OUT_SILU (and likewise OUT_CLIP with its own product): Wp is the fused [2 I, K] gate / up matrix (N = 2 I, gate rows first) and the output is
// act = silu(elt(gate)) * elt(up) [T, I] in fragment order (tiles per 32-k step: x_tt).  A block is 256 tokens x 128
// channels: the ring slots of a stage hold, for each of the two row groups of waves, four gate tiles and then the four
// up tiles of the same channels, so that a lane ends up with both halves of its channels and the product never leaves
// the registers.  LoRA deltas: slot 0 of `lo` is the gate projection, slot 1 the up projection (B == nullptr: not
// adapted); each rides as its own extra k-steps, in which only that half of a wave's tiles is multiplied.
// LORA = false is the plain GEMM (lo is ignored); GROUPED: see PPGroup (gy is the number of tiles in use)
template <int OUT, bool LORA, bool GROUPED = false>
__global__ __launch_bounds__(PP_WAVES* WAVE, 2) void gemm_pp_kernel(void* __restrict__ yv, const elt* __restrict__ x, int ldx, int x_tt,
                                                                   const elt* __restrict__ Wp, int T, int K, int N, int gx, int gy,
                                                                   PPLora lo, GluArgs ga, PPGroup gr = PPGroup()) {
  if constexpr (GROUPED) gy = *gr.plan.n_tiles;
  extern __shared__ __align__(16) elt smem[];  // [PP_STAGES][PP_STAGE_ELEMS], then [PP_WAVES][PP_OUT_ELEMS]
  constexpr int NW = PP_WAVES;
  constexpr int LQ = 2 * PP_F / NW;            // fragments a wave fetches per stage (4)
  constexpr int WTF = 4;                       // token fragments of a wave's tile (64 tokens)
  constexpr bool SILU = OUT == OUT_SILU || OUT == OUT_CLIP;   // a gated product
  constexpr int BN = SILU ? PP_F * 8 : PP_F * 16;   // output columns of a block (SILU: channels, each a gate and an up row)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int nb = gx * gy;
  const int KB = K / 32;
  const int tiles = (N + 15) / 16;
  const int I = N / 2, itiles = I / 16;        // SILU: channels and their 16-row tiles
  const int G = gridDim.x;
  if constexpr (GROUPED) {
    if ((int)blockIdx.x >= nb) return;         // fewer blocks than workgroups: nothing was requested yet
  }

  // Block number -> (weight-row block, token block).  Each XCD takes an eighth of the blocks, in their order: bands of BAND
  // token blocks, within a band all token blocks of a weight-row block before those of the next.  So the 32 blocks that an XCD
  // multiplies at a time are some token blocks times some weight-row blocks and share both in its L2, where all token blocks of
  // one weight-row block shared only that.  Bands of 4 against one band, fragment-ordered x: 4001 tokens x 22016 x 4096 653 -> 614 us,
  // 8192 tokens 1301 -> 1150, 8192 tokens x 4096 x 11008 611 -> 552, 2500 x 12288 x 4096 190 -> 189; 8 is within 1 %, 2 to 3 % slower
  // on 22016 rows.  Row-major x, 64 bytes of 16 rows per fragment, keeps one band (4: 3000 x 12288 x 4096 305 -> 323 us).  Over a
  // plan a band of 3 tiles has most of an expert's tiles together (32 experts of 5504 x 4096, uniform plans alone, 8000 tokens of 4: 1660 us
  // in one band, 1585 with 3 or 4, 1592 with 8; 4000 tokens 912, 892, 902, 910).  In whole passes, where runs
  // differ by 0.2 to 0.4 %, one band, 4 and 8 take as long as 3 and 1.3 %, -0.1 %, 0.4 % (Dinasun over 4001 tokens), 0.6 %, 0.5 %, 0.2 %
  // (Safolorn over 3683) more.
  constexpr unsigned BAND = GROUPED ? 3 : 4;
  auto block_of = [&](int L, int& n0, int& t0) {
    const unsigned xcd = L & 7, more = nb & 7;
    const unsigned idx = xcd * (nb >> 3) + (xcd < more ? xcd : more) + (L >> 3);
    unsigned first = 0, r = idx, h = gy, row;
    if (GROUPED || x_tt > 0) {
      first = idx / (BAND * gx) * BAND;        // the only division by a number that is not a constant: they take longer than a k-step
      r -= first * gx;
      h = gy - first < BAND ? gy - first : BAND;
      row = h == 4 ? r / 4 : h == 3 ? r / 3 : h == 2 ? r / 2 : r;
    } else {
      row = r / h;
    }
    n0 = row * BN;
    t0 = first + r - row * h;
    if constexpr (GROUPED) t0 = __builtin_amdgcn_readfirstlane(t0);      // a tile of the plan
    else t0 *= PP_F * 16;
  };
  // the LoRA part of a block: projection slot and adapter (-1: none), everything uniform
  auto lora_of = [&](int n0, int t0, int& slot) -> int {
    // (through the constant cache: a vector load would wait behind everything that is on its way to LDS)
    const auto adapter_of = [&](int t0) { return ((const __attribute__((address_space(4))) int32_t*)lo.blk_adapter)[__builtin_amdgcn_readfirstlane(t0) / (PP_F * 16)]; };
    if constexpr (SILU) {
      slot = 0;
      return adapter_of(t0);
    }
    slot = -1;
#pragma unroll
    for (int i = 0; i < 3; ++i)
      if (i < lo.n_proj && n0 >= lo.n_begin[i] && n0 < lo.n_begin[i] + lo.n_rows[i]) slot = i;
    if (slot < 0) return -1;
    return adapter_of(t0);
  };
  auto tile_of = [&](int i) { return ((const __attribute__((address_space(4))) i32x4*)gr.plan.tiles)[i]; };   // i uniform: through the constant cache, a vector load would wait behind everything on its way to LDS
  auto pick = [](int i, auto a, auto b, auto c) { return i == 0 ? a : i == 1 ? b : c; };   // by value: `lo` is never indexed by a variable
  const int EP = LORA ? 2 * (lo.r / 32) : 0;    // extra k-steps per projection of a block with a delta: hi halves, then lo halves
  const bool has_gate = SILU && LORA && lo.B[0] != nullptr;
  const int E = SILU ? EP * ((lo.B[0] != nullptr) + (lo.B[1] != nullptr)) : EP;

  // ---- loader role: wave w fetches fragments 4 w .. 4 w + 3 of every stage (waves 0-3: weights, waves 4-7: tokens)
  const elt* src[LQ];
  int step = 0;                                // elements between consecutive k-steps of this wave's sources
  int load_L = blockIdx.x, load_kb = 0;        // the stage the loader issues next
  int load_nst = KB;                           // stages of the block being loaded (KB, or KB + E with a delta)
  const elt* l_src = nullptr;                  // LoRA stages of that block (all uniform): row 0 of the block in B[a] (weight waves) or in v_hi (token waves) ...
  long l_lo = 0;                               // ... the distance from v_hi to v_lo (token waves; 0 for weight waves) ...
  int l_rows = 1;                              // ... and the rows that exist from there on (rows past them repeat the last one; their results are dropped)
  int l_a = -1, l_n0 = 0, l_t0 = 0;            // SILU: adapter, first channel and first token of that block (the stages' addresses are formed per stage)
  auto load_block = [&](int L) {
    int n0, t0;
    block_of(L < nb ? L : blockIdx.x, n0, t0); // past the last block: valid addresses, the data is never multiplied
    load_nst = KB;
    const elt* Wb = Wp;
    int last_tt = x_tt - 1;                    // tiles past it: a valid fragment, results dropped (of a plan's tile its own last one, at hand already)
    if constexpr (GROUPED) {
      const i32x4 tile = tile_of(t0);
      Wb = Wp + __builtin_amdgcn_readfirstlane(tile.x) * gr.w_elems;
      t0 = __builtin_amdgcn_readfirstlane(tile.y);
      last_tt = (t0 + __builtin_amdgcn_readfirstlane(tile.z) - 1) / 16;
    }
    if constexpr (LORA) {
      int slot;
      const int a = L < nb ? lora_of(n0, t0, slot) : -1;
      if (a >= 0) load_nst = __builtin_amdgcn_readfirstlane(KB + E);
      if (SILU) {
        l_a = a;
        l_n0 = n0;
        l_t0 = t0;
      } else if (a >= 0) {
        const elt* Bt = pick(slot, lo.B[0], lo.B[1], lo.B[2]);
        const elt* vh = pick(slot, lo.vh[0], lo.vh[1], lo.vh[2]);
        const elt* vl = pick(slot, lo.vl[0], lo.vl[1], lo.vl[2]);
        const int nbeg = pick(slot, lo.n_begin[0], lo.n_begin[1], lo.n_begin[2]), nrows = pick(slot, lo.n_rows[0], lo.n_rows[1], lo.n_rows[2]);
        if (wave < NW / 2) {
          l_src = Bt + ((size_t)a * nrows + (n0 - nbeg)) * lo.r;
          l_lo = 0;
          l_rows = nrows - (n0 - nbeg);
        } else {
          l_src = vh + (size_t)t0 * lo.r;
          l_lo = vl - vh;
          l_rows = T - t0;
        }
        // all of this is the same in every lane: say so, it lives in scalar registers across the K loop
        l_src = (const elt*)uniform64((unsigned long long)l_src);
        l_lo = (long)uniform64((unsigned long long)l_lo);
        l_rows = __builtin_amdgcn_readfirstlane(l_rows);
      }
    }
    if (wave < NW / 2) {
#pragma unroll
      for (int q = 0; q < LQ; ++q) {
        int nt;
        if constexpr (SILU) {                  // slots 8 wn + 0..3: gate tiles of channels n0 + 64 wn .., slots 8 wn + 4..7: their up tiles
          int it = n0 / 16 + (wave >> 1) * LQ + q;
          it = it < itiles ? it : itiles - 1;
          nt = it + (wave & 1) * itiles;
        } else {
          nt = n0 / 16 + wave * LQ + q;
          nt = nt < tiles ? nt : tiles - 1;    // rows past N: a valid fragment, results dropped
        }
        src[q] = Wb + (size_t)nt * KB * 512 + lane * 8;
      }
      step = 512;
    } else if (x_tt > 0) {
#pragma unroll
      for (int q = 0; q < LQ; ++q) {
        int tt = t0 / 16 + (wave - NW / 2) * LQ + q;
        tt = tt < last_tt ? tt : last_tt;
        src[q] = x + (size_t)tt * 512 + lane * 8;
      }
      step = x_tt * 512;
    } else {
#pragma unroll
      for (int q = 0; q < LQ; ++q) {
        int t = t0 + ((wave - NW / 2) * LQ + q) * 16 + (lane & 15);
        t = t < T ? t : T - 1;
        src[q] = x + (size_t)t * ldx + (lane >> 4) * 8;
      }
      step = 32;
    }
  };
  int ring = 0;                                // ring slot of the stage issued next
  // PLAIN: the caller knows that this stage is an ordinary k-step and not the last of its block (no tests at all)
  auto issue = [&](auto PLAIN) {
    constexpr bool plain = decltype(PLAIN)::value;
    elt* dst = smem + ring * PP_STAGE_ELEMS + wave * LQ * 512;
    if (plain || !LORA || load_kb < KB) {
#pragma unroll
      for (int q = 0; q < LQ; ++q)
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src[q] + (size_t)load_kb * step),
                                         (__attribute__((address_space(3))) void*)(dst + q * 512), 16, 0, 0);
    } else if constexpr (SILU) {               // a LoRA stage of the gate or of the up projection
      const int j = load_kb - KB, RB = lo.r / 32;
      const bool up = !(has_gate && j < EP);   // uniform
      const int jj = has_gate && up ? j - EP : j;
      const bool lo_half = jj >= RB;
      const int ks = (lo_half ? jj - RB : jj) * 32;
      const elt* base;
      int row0, rows;
      if (wave < NW / 2) {                     // rows of the projection's table for this wave's channels (used by the waves of that half only)
        base = (up ? lo.B[1] : lo.B[0]) + (size_t)l_a * I * lo.r;
        row0 = l_n0 + (wave >> 1) * (LQ * 16);
        rows = I;
      } else {
        base = up ? (lo_half ? lo.vl[1] : lo.vh[1]) : (lo_half ? lo.vl[0] : lo.vh[0]);
        row0 = l_t0 + (wave & 3) * (LQ * 16);
        rows = T;
      }
#pragma unroll
      for (int q = 0; q < LQ; ++q) {
        int row = row0 + q * 16 + (lane & 15);
        row = row < rows ? row : rows - 1;
        const elt* p = base + ((size_t)row * lo.r + ks + (lane >> 4) * 8);
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)p,
                                         (__attribute__((address_space(3))) void*)(dst + q * 512), 16, 0, 0);
      }
    } else {                                   // a LoRA stage: 16 rows x 64 bytes per fragment, gathered by the lanes' addresses
      const int j = load_kb - KB, RB = lo.r / 32;
      const int ks = (j < RB ? j : j - RB) * 32;
#pragma unroll
      for (int q = 0; q < LQ; ++q) {
        int row = ((wave & 3) * LQ + q) * 16 + (lane & 15);
        row = row < l_rows ? row : l_rows - 1;
        const elt* p = l_src + (j < RB ? 0 : l_lo) + ((size_t)row * lo.r + ks + (lane >> 4) * 8);
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)p,
                                         (__attribute__((address_space(3))) void*)(dst + q * 512), 16, 0, 0);
      }
    }
    ring = (ring + 1) & (PP_STAGES - 1);
    ++load_kb;
    if constexpr (!plain) {
      if (load_kb == load_nst) {               // uniform
        load_kb = 0;
        load_L += G;
        load_block(load_L);
      }
    }
  };

  // ---- compute role: rows wn * 128 .., tokens wt * 64 ..
  // (a group has 128 of the weight rows, a SIMD's two waves the two halves)
  const int wn = wave / (NW / 2), wt = wave & 3;
  f32x4 acc[8][WTF];
  eltx8 a[8], b[WTF];
  int rd = 0;                                  // ring slot of the stage whose fragments are read next
  // The token fragments of a wave: four in a row; of a plan's tile every fourth, so that the places a tile does have - often few of
  // its 256 - spread over all waves, and the first `have` of them are multiplied (uniform; the others are fetched and read like them, but
  // their accumulators never stored).
  auto tfrag = [&](int j) { return GROUPED ? wt + 4 * j : wt * WTF + j; };
  // First half of a stage: this wave's fragments from LDS into registers, its share of the stage three ahead on its way into the slot
  // that all waves have done with, and the wait for its share of the next stage (at most the two stages after that still in flight).
  auto fetch = [&](auto PLAIN) {
    const elt* st = smem + rd * PP_STAGE_ELEMS + lane * 8;
#pragma unroll
    for (int j = 0; j < WTF; ++j) b[j] = ld8(st + (PP_F + tfrag(j)) * 512);
#pragma unroll
    for (int i = 0; i < 8; ++i) a[i] = ld8(st + (wn * 8 + i) * 512);
    rd = (rd + 1) & (PP_STAGES - 1);
    issue(PLAIN);
    asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    bare_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  // Second half: the products.  half (uniform): -1 all eight row tiles, 0 / 1 the first / last four (a LoRA stage of the gate / up
  // projection).  The barrier at its end lets the other group begin: ahead of the last four or eight products, to cover its latency, it
  // has both groups multiply at once and costs 10 % (4096 x 12288 x 4096 287 -> 314 us).
  auto multiply = [&](int half, int have) {
    __builtin_amdgcn_s_setprio(1);
    if constexpr (GROUPED) {
      asm volatile("" : "+s"(have));           // compared where it is used, in scalar registers
#pragma unroll
      for (int j = 0; j < WTF; ++j)
        if (__builtin_expect(j < have, 1)) {   // uniform; the products of a full tile follow each other without a jump
#pragma unroll
          for (int i = 0; i < 8; ++i) acc[i][j] = mfma_16x16x32(a[i], b[j], acc[i][j]);
        }
    } else {
      if (half != 1) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < WTF; ++j) acc[i][j] = mfma_16x16x32(a[i], b[j], acc[i][j]);
      }
      if (half != 0) {
#pragma unroll
        for (int i = 4; i < 8; ++i)
#pragma unroll
          for (int j = 0; j < WTF; ++j) acc[i][j] = mfma_16x16x32(a[i], b[j], acc[i][j]);
      }
    }
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
    bare_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };

  load_block(load_L);
  issue(std::false_type());
  issue(std::false_type());
  issue(std::false_type());
  asm volatile("s_waitcnt vmcnt(8)" ::: "memory");     // the first stage of this wave has landed
  bare_barrier();
  elt* ostage = smem + PP_STAGES * PP_STAGE_ELEMS + wave * PP_OUT_ELEMS;
  const int r16 = lane & 15, g = lane >> 4;
  for (int L = blockIdx.x; L < nb; L += G) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < WTF; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    int n0, t0;
    block_of(L, n0, t0);
    int tend = T, have = WTF;
    if constexpr (GROUPED) {
      const i32x4 tile = tile_of(t0);
      t0 = __builtin_amdgcn_readfirstlane(tile.y);
      tend = t0 + __builtin_amdgcn_readfirstlane(tile.z);
      have = tend - t0 <= wt * 16 || (SILU ? n0 + wn * 64 >= I : n0 + wn * 128 >= N) ? 0 : (tend - t0 - wt * 16 + 63) / 64;
    }
    int nst = KB;
    if constexpr (LORA) {
      int slot;
      if (lora_of(n0, t0, slot) >= 0) nst += E;
      nst = __builtin_amdgcn_readfirstlane(nst);
    }
    // While ordinary k-steps of one block are fetched and multiplied nothing is tested; the last stages of a block and those of a
    // delta take the general form.
    int kb = KB - 1 - load_kb;
    kb = kb < 0 ? 0 : kb;
    if (wave >= NW / 2) bare_barrier();        // the second group: half a stage behind the first
    for (int left = kb; left > 0; --left) {
      fetch(std::true_type());
      multiply(-1, have);
    }
    for (; kb < nst; ++kb) {
      const int half = !(SILU && LORA) || kb < KB ? -1 : (has_gate && kb - KB < EP ? 0 : 1);   // uniform
      fetch(std::false_type());
      multiply(half, have);
    }
    // Both groups store together; half a stage apart each waited for the other's memory rounds: 4096 x 12288 x 4096 in bf16, three rounds
    // of blocks, with a gated product 290 -> 285 us; in fp16 added to fp32 379 -> 351, 4096 x 4096 x 4096 115 -> 112, 2800 x 256 x 9824 56 -> 48.
    if (wave < NW / 2) bare_barrier();
    if constexpr (SILU) {
      // acc[i] and acc[4 + i] are the gate and the up half of channels n0 + wn * 64 + i * 16 + 4 g .. + 3 for token r16 of
      // token fragment j: four products = one 8-byte piece of the output fragment; the pieces of a store instruction
      // are 512 contiguous bytes
#pragma unroll
      for (int j = 0; j < WTF; ++j) {
        const int t = t0 + tfrag(j) * 16 + r16;
        if ((t >> 4) >= x_tt || (GROUPED && t >= tend)) continue;   // the token tile does not exist (the place is another expert's)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int c = n0 + (wn * 4 + i) * 16 + g * 4;
          if (c >= I) continue;
          eltx4 o = eltx4{0, 0, 0, 0};                   // rows past T inside the last tile: zeros, as the separate kernel writes them
          if (t < T) {
#pragma unroll
            for (int r = 0; r < 4; ++r) o[r] = (elt)glu<OUT == OUT_CLIP ? MLORA_GLU_CLIPPED : MLORA_GLU_SILU>(acc[i][j][r], acc[4 + i][j][r], ga);
          }
          *reinterpret_cast<eltx4*>((elt*)yv + ((size_t)(c >> 5) * x_tt + (t >> 4)) * 512 + ((c & 31) >> 3) * 128 + (t & 15) * 8 + (c & 7)) = o;
        }
      }
    } else if constexpr (OUT == OUT_RELU2) {
      // four channels of a token = one 8-byte piece of the output fragment
#pragma unroll
      for (int j = 0; j < WTF; ++j) {
        const int t = t0 + tfrag(j) * 16 + r16;
        if (t >= tend) continue;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int c = n0 + (wn * 8 + i) * 16 + g * 4;
          if (c >= N) continue;
          eltx4 o;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float v = fmaxf(acc[i][j][r] * gr.alpha, 0.f);
            o[r] = (elt)(v * v);
          }
          *reinterpret_cast<eltx4*>((elt*)yv + ((size_t)(c >> 5) * x_tt + (t >> 4)) * 512 + ((c & 31) >> 3) * 128 + (t & 15) * 8 + (c & 7)) = o;
        }
      }
    } else if constexpr (OUT == OUT_F16) {
      // 16 tokens x 64 columns at a time through the wave's staging buffer: D[n][t] fragments in, token rows out
      int rows[WTF][2];                                // requested together
#pragma unroll
      for (int j = 0; j < WTF; ++j)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          rows[j][q] = t0 + tfrag(j) * 16 + q * 8 + (lane >> 3);
          if constexpr (GROUPED) rows[j][q] = gr.plan.perm[rows[j][q] < tend ? rows[j][q] : tend - 1];
        }
#pragma unroll
      for (int j = 0; j < WTF; ++j) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            f32x4 sacc = acc[h * 4 + i][j];
            if constexpr (GROUPED) sacc *= gr.alpha;
            *reinterpret_cast<eltx4*>(ostage + r16 * PP_OUT_LD + i * 16 + g * 4) = eltx4{(elt)sacc[0], (elt)sacc[1], (elt)sacc[2], (elt)sacc[3]};
          }
          __builtin_amdgcn_wave_barrier();
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            const int c = q * 64 + lane;           // 16-byte chunk: token row c / 8, columns (c % 8) * 8 ..
            const int tr = c >> 3, cc = (c & 7) * 8;
            const int t = t0 + tfrag(j) * 16 + tr;
            const int row = rows[j][q];
            const int n = n0 + (wn * 8 + h * 4) * 16 + cc;
            const eltx4 lo = *reinterpret_cast<const eltx4*>(ostage + tr * PP_OUT_LD + cc);
            const eltx4 hi = *reinterpret_cast<const eltx4*>(ostage + tr * PP_OUT_LD + cc + 4);
            if (t < tend && n + 8 <= N) {
              st8((elt*)yv + (size_t)row * N + n, eltx8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
            } else if (t < tend) {
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                if (n + e < N) ((elt*)yv)[(size_t)row * N + n + e] = lo[e];
                if (n + 4 + e < N) ((elt*)yv)[(size_t)row * N + n + 4 + e] = hi[e];
              }
            }
          }
          __builtin_amdgcn_wave_barrier();
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < WTF; ++j) {
        const int t = t0 + tfrag(j) * 16 + r16;
        if (t >= T) continue;
        // Added to fp32: each value is read right ahead of its store.  A token's eight requested together leave the compute unit's memory idle while
        // they are added: fp16, 2800 x 256 x 9824 47.5 -> 51.6 us, 3450 x 512 x 4096 32.1 -> 34.6, 3571 x 2048 x 4096 63.2 -> 65.4, 3219 x 11008 x 4096 235 -> 232;
        // only rows of 12288 gain by it (2338 x 1408 100.7 -> 102.7, but 4297 x 4096 434 -> 424).
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int n = n0 + (wn * 8 + i) * 16 + g * 4;        // N is a multiple of 4 (checked)
          if (n >= N) continue;
          f32x4* p = reinterpret_cast<f32x4*>((float*)yv + (size_t)t * N + n);
          if constexpr (OUT == OUT_ACC_F32) *p = *p + acc[i][j];
          else *p = acc[i][j];
        }
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // the loads issued past the last block must not outlive the workgroup's LDS
}

template <int OUT>
int launch_gemm_pp(void* y, const elt* x, int ldx, int x_tt, const elt* Wp, int T, int K, int N, hipStream_t s,
                   const PPLora& lo = PPLora(), const GluArgs& ga = GluArgs()) {
  constexpr size_t lds = ((size_t)PP_STAGES * PP_STAGE_ELEMS + (size_t)PP_WAVES * PP_OUT_ELEMS) * sizeof(elt);
  // the attribute is per kernel, set once per process (the initialiser of a local static runs once, also when several
  // host threads make their first call together)
  static const hipError_t configured = [] {
    hipError_t e = hipFuncSetAttribute((const void*)gemm_pp_kernel<OUT, false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e == hipSuccess) e = hipFuncSetAttribute((const void*)gemm_pp_kernel<OUT, OUT != OUT_CLIP>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    return e;
  }();
  if (configured != hipSuccess)
    return mlora_set_error(MLORA_ERR_LAUNCH, "gemm_packed: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(configured));
  const int gx = OUT == OUT_SILU || OUT == OUT_CLIP ? ceil_div(N / 2, PP_F * 8) : ceil_div(N, PP_F * 16), gy = ceil_div(T, PP_F * 16);
  int n_cu = gemm_n_cu();
  if (n_cu <= 0) n_cu = 256;
  const int grid = gx * gy < n_cu ? gx * gy : n_cu;
  if (lo.n_proj > 0 && OUT != OUT_CLIP) hipLaunchKernelGGL((gemm_pp_kernel<OUT, OUT != OUT_CLIP>), dim3(grid), dim3(PP_WAVES * WAVE), lds, s, y, x, ldx, x_tt, Wp, T, K, N, gx, gy, lo, ga);
  else hipLaunchKernelGGL((gemm_pp_kernel<OUT, false>), dim3(grid), dim3(PP_WAVES * WAVE), lds, s, y, x, ldx, x_tt, Wp, T, K, N, gx, gy, lo, ga);
  return MLORA_OK;
}

// ---------------------------------------------------------------------------------------------
// Products between the decode GEMV and the persistent kernel above (from 65 tokens on: a decode step of many sequences, a
// short prefill, and what does not fill whole rounds of the kernel above).  The matrix cores, LDS and the operand loads
// weigh about the same, so the block is chosen by size (gemm_mid_shape): FT x FN fragments (128, 192 or 256 tokens x 128, 96 or
// 64 weight rows), eight waves, both operands in fragment
// order and copied from global memory straight into an LDS ring.  A stage of the ring is TWO 32-k steps: with the
// few MFMAs a wave has per 32-k step here (4 to 16), a barrier and a wait per step cost more than the step itself.
// Four (three) stages, of which three (two) are in flight per compute unit - across the barrier of a stage, which is
// the bare instruction (bare_barrier): behind __syncthreads() the compiler first waits for every request in flight,
// the ring ran as if it had one stage and the launch pulled 2 to 3.4 TB/s of weights whatever its depth.
// What bounds the kernel is LDS: per stage of 256 x 96 the waves read 112 KiB of fragments and the loads bring 44 KiB, at 128
// bytes a cycle, beside 768 cycles of products per SIMD; so the reads go out between the products (3 to 9 % of a launch over reads
// ahead of them: gate/up at 137 tokens 61.7 -> 56.6 us).  It is neither the second-level caches (a compute unit can take in 130 GB/s
// of hits, the kernel asks for 45) nor the depth of the ring (a ring of seven weight stages beside three of tokens was 2 to 5 %
// slower).  So a wave whose tokens all lie past T reads and multiplies nothing, which leaves its share of LDS to the others:
// 137 tokens x 12288 x 4096 32.5 -> 29.0 us, 270 x 22016 x 4096 89.6 -> 80.2, 400 x 22016 80.8 -> 77.3.  (The fragments past T are
// still loaded: dealing only the others out to the waves, each waiting for a count of its own, took more than it saved, 29.0 -> 32 to 36.)
// grid = (weight-row blocks, K slices, token blocks).
// With K slices, slice 0 produces the result proper (store or accumulate) and slice s > 0 stores its fp32 partial
// sums to part[s - 1][T][ld_part] - for the two narrow accumulating linears of a layer, whose partials the next
// RMSNorm of the row adds in slice order.
// ---------------------------------------------------------------------------------------------
constexpr int MID_KS = 2;                      // 32-k steps per stage
constexpr int mid_stages(int FT) { return FT == 16 ? 3 : 4; }

// LORA: the deltas of any mix of adapters (linear_add_deltas) come into the accumulators ahead of the first step, while the ring fills.  Behind
// the last step, as further steps of the ring, the same took 11 us: cold code and addresses that nothing hides.  137 tokens of one adapter of rank
// 16, us: q, k, v (K 4096, N 12288) linear 31.0, shrink 5.4, expand 7.7 -> shrink 6.4, linear 37.8; o (N 4096, four K slices) 15.6, 5.0, 8.3 -> 6.4, 19.2.
// GX: the rows are groups of gx_rows (a multiple of 16 FN) that read activations of their own, gx_stride elements apart.
// A gated product (OUT_SILU, OUT_CLIP): Wp is the fused [2 I, K] matrix (N = 2 I), a block FN / 2 tiles of gate rows and the up rows of the same
// channels, so that the waves wn = 0 hold the one and wn = 1 the other; they exchange halves through LDS, rounded to elements as a linear
// would store them, and leave the product in fragment order.
template <int OUT, int FT, int FN, bool GX = false, bool LORA = false>
__global__ __launch_bounds__(PP_WAVES* WAVE, 2) void gemm_mid_kernel(void* __restrict__ yv, float* __restrict__ part, int ld_part,
                                                                    const elt* __restrict__ xf, int x_tt, const elt* __restrict__ Wp,
                                                                    int T, int K, int N, int gx_rows = 0, long gx_stride = 0,
                                                                    GluArgs ga = GluArgs(), LinearDeltas lo = LinearDeltas()) {
  constexpr bool GLU = OUT == OUT_SILU || OUT == OUT_CLIP;
  constexpr int MID_STAGES = mid_stages(FT);
  constexpr int SF = FN + FT;                  // fragments of one 32-k step: weights, then tokens
  constexpr int LF = MID_KS * SF;              // fragments per stage
  constexpr int LQ = (LF + PP_WAVES - 1) / PP_WAVES;   // ... of which a wave fetches LQ (fragment f = wave + 8 q: fragment f % SF of k-step f / SF)
  constexpr int LREM = LF % PP_WAVES;          // ... or, when they do not divide, the waves from LREM on one fewer
  constexpr int STAGE_ELEMS = LF * 512;
  constexpr int WTF = FT / 4;                  // token fragments of a wave's tile
  constexpr int WNF = FN / 2;                  // weight fragments of a wave's tile
  constexpr int VM = (MID_STAGES - 2) * LQ;    // a wave's loads that may still be in flight when the next stage is read
  constexpr int VM1 = (MID_STAGES - 2) * (LQ - 1);   // ... for the waves with one fragment fewer
  static_assert(FT % 4 == 0 && FN % 2 == 0 && WNF <= 4, "the tile divides over the waves");
  extern __shared__ __align__(16) elt smem[];  // [MID_STAGES][STAGE_ELEMS]; the output staging reuses it after the K loop
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int KB = K / 32;
  const int tiles = (N + 15) / 16;
  const int n0 = blockIdx.x * FN * (GLU ? 8 : 16), t0 = blockIdx.z * FT * 16;       // GLU: the first channel
  const int I = N / 2, itiles = I / 16;
  auto tile_row = [&](int f) {                 // the 16-row tile of W that is weight fragment f of the block (it may lie past the end)
    if constexpr (GLU) return f < FN / 2 ? n0 / 16 + f : itiles + n0 / 16 + f - FN / 2;
    return n0 / 16 + f;
  };
  if constexpr (GX) xf += (n0 / gx_rows) * gx_stride;
  const int per = (KB + gridDim.y - 1) / gridDim.y;
  const int kb0 = blockIdx.y * per;
  const int kb1 = kb0 + per < KB ? kb0 + per : KB;
  const int nks = kb1 - kb0;                   // 32-k steps of this slice (>= 1: checked by the launcher)
  const int nst = (nks + MID_KS - 1) / MID_KS; // stages

  const elt* src[LQ];
  int step[LQ], kso[LQ];
#pragma unroll
  for (int q = 0; q < LQ; ++q) {
    const int f = (wave + PP_WAVES * q) % SF;  // uniform (past LF for the last q of a wave with one fewer: set up, never issued)
    kso[q] = (wave + PP_WAVES * q) / SF;
    if (f < FN) {
      int nt = tile_row(f);
      nt = nt < tiles ? nt : tiles - 1;        // rows past N: a valid fragment, results dropped (past the gate's: the up part's first ones)
      src[q] = Wp + (size_t)nt * KB * 512 + lane * 8;
      step[q] = 512;
    } else {
      int tt = t0 / 16 + f - FN;
      tt = tt < x_tt ? tt : x_tt - 1;          // tiles past T: a valid fragment, results dropped
      src[q] = xf + (size_t)tt * 512 + lane * 8;
      step[q] = x_tt * 512;
    }
  }
  int ring = 0, load_kb = kb0;
  auto issue = [&]() {
    elt* dst = smem + ring * STAGE_ELEMS + wave * 512;
#pragma unroll
    for (int q = 0; q < LQ; ++q) {
      if (LREM != 0 && q == LQ - 1 && wave >= LREM) break;      // uniform
      int kb = load_kb + kso[q];
      kb = kb < kb1 ? kb : kb1 - 1;            // past the slice: a valid address; the data is not multiplied
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src[q] + (size_t)kb * step[q]),
                                       (__attribute__((address_space(3))) void*)(dst + q * PP_WAVES * 512), 16, 0, 0);
    }
    ring = ring + 1 == MID_STAGES ? 0 : ring + 1;
    load_kb += MID_KS;
  };

  const int wn = wave & 1, wt = wave >> 1;     // weight rows wn * WNF * 16 .., tokens wt * WTF * 16 ..
  f32x4 acc[WNF][WTF];
  eltx8 a[2][MID_KS][WNF], b[2][MID_KS][WTF];  // two register sets: the stage being multiplied and its successor
#pragma unroll
  for (int i = 0; i < WNF; ++i)
#pragma unroll
    for (int j = 0; j < WTF; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  int rd = 0;
  auto read_frags = [&](auto U) {
    constexpr int u = decltype(U)::value;
    const elt* st = smem + rd * STAGE_ELEMS + lane * 8;
#pragma unroll
    for (int ks = 0; ks < MID_KS; ++ks) {
#pragma unroll
      for (int j = 0; j < WTF; ++j) b[u][ks][j] = ld8(st + (ks * SF + FN + wt * WTF + j) * 512);
#pragma unroll
      for (int i = 0; i < WNF; ++i) a[u][ks][i] = ld8(st + (ks * SF + wn * WNF + i) * 512);
    }
    rd = rd + 1 == MID_STAGES ? 0 : rd + 1;
  };
  int done_ks = 0;                             // 32-k steps multiplied so far
  auto multiply = [&](auto U) {
    constexpr int u = decltype(U)::value;
#pragma unroll
    for (int ks = 0; ks < MID_KS; ++ks) {
      if (done_ks + ks < nks) {                // uniform: the last stage of an odd slice holds one step only
#pragma unroll
        for (int i = 0; i < WNF; ++i)
#pragma unroll
          for (int j = 0; j < WTF; ++j) acc[i][j] = mfma_16x16x32(a[u][ks][i], b[u][ks][j], acc[i][j]);
      }
    }
    done_ks += MID_KS;
  };
  // the wait: of this wave's loads at most those of the MID_STAGES - 2 youngest stages are still in flight, so the
  // stage multiplied next has landed; with everybody's wait and fragment reads behind the barrier, the slot of the
  // stage just read is refilled
  auto wait_next = [&]() {
    if (LREM != 0 && wave >= LREM) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(VM1) : "memory");       // uniform
    else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(VM) : "memory");
  };
  // A stage: the fragment reads of its successor go out between its products.  All at once ahead of them, the reads of eight
  // waves (8 - 16 KiB each, 128 bytes a cycle) hold up the first product by as long as the products take.
  auto stage = [&](auto U, auto WHOLE) {
    constexpr int u = decltype(U)::value;
    wait_next();
    bare_barrier();
    issue();
    if constexpr (decltype(WHOLE)::value) {
      constexpr int NP = MID_KS * WNF * WTF, NR = MID_KS * (WNF + WTF), SPAN = NP * 3 / 4;
      const elt* st = smem + rd * STAGE_ELEMS + lane * 8;
      rd = rd + 1 == MID_STAGES ? 0 : rd + 1;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        const int ks = p / (WNF * WTF), i = p / WTF % WNF, j = p % WTF;
        acc[i][j] = mfma_16x16x32(a[u][ks][i], b[u][ks][j], acc[i][j]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = p * NR / SPAN; r < (p + 1) * NR / SPAN && r < NR; ++r) {
          const int rs = r / (WNF + WTF), f = r % (WNF + WTF);
          if (f < WTF) b[1 - u][rs][f] = ld8(st + (rs * SF + FN + wt * WTF + f) * 512);
          else a[1 - u][rs][f - WTF] = ld8(st + (rs * SF + wn * WNF + f - WTF) * 512);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      done_ks += MID_KS;
    } else {
      read_frags(std::integral_constant<int, 1 - u>());
      __builtin_amdgcn_sched_barrier(0);
      multiply(U);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  int left[LORA ? WTF : 1];                    // the adapters of this lane's tokens that are still to be done: asked for ahead of the ring's loads
  if constexpr (LORA) {
#pragma unroll
    for (int j = 0; j < WTF; ++j) {
      const int t = t0 + (wt * WTF + j) * 16 + (lane & 15);
      left[j] = t < T ? lo.ids[t] : -1;
    }
  }
#pragma unroll
  for (int i = 0; i < MID_STAGES - 1; ++i) issue();
  if constexpr (LORA) {
    if (blockIdx.y == 0 && t0 + wt * WTF * 16 < T) {             // uniform: slice 0, a wave with tokens
      int row0[WNF];
#pragma unroll
      for (int i = 0; i < WNF; ++i) row0[i] = tile_row(wn * WNF + i) * 16;
      int half[WTF];
      linear_add_deltas<WNF, WTF, false>(acc, lo, left, half, T, t0 + wt * WTF * 16, row0, lane, 0, 1);
    }
  }
  wait_next();
  bare_barrier();
  issue();
  if (t0 + wt * WTF * 16 >= T) {               // uniform: no token of this wave exists; it only takes its part in the loads
    for (int s = 0; s < nst; ++s) {
      wait_next();
      bare_barrier();
      issue();
    }
  } else {
    read_frags(std::integral_constant<int, 0>());
    int g = 0;
    const int whole = nks / MID_KS;            // stages of two steps; an odd slice ends in one of a single step
    for (; g + 1 < whole; g += 2) {
      stage(std::integral_constant<int, 0>(), std::true_type());
      stage(std::integral_constant<int, 1>(), std::true_type());
    }
    if (g < nst) stage(std::integral_constant<int, 0>(), std::false_type());
    if (g + 1 < nst) stage(std::integral_constant<int, 1>(), std::false_type());
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");   // nothing is in flight into the LDS that the epilogue reuses
  __syncthreads();

  const int r16 = lane & 15, gq = lane >> 4;
  if (blockIdx.y > 0) {                        // a later K slice: fp32 partial sums
    float* pp = part + (size_t)(blockIdx.y - 1) * T * ld_part;
#pragma unroll
    for (int j = 0; j < WTF; ++j) {
      const int t = t0 + (wt * WTF + j) * 16 + r16;
      if (t >= T) continue;
#pragma unroll
      for (int i = 0; i < WNF; ++i) {
        const int n = n0 + (wn * WNF + i) * 16 + gq * 4;
        if (n < N) *reinterpret_cast<f32x4*>(pp + (size_t)t * ld_part + n) = acc[i][j];
      }
    }
    return;
  }
  if constexpr (GLU) {
    // waves wn = 0 finish the first token fragments of a pair of waves, wn = 1 the others
    constexpr int H0 = (WTF + 1) / 2;
    eltx4* ex = reinterpret_cast<eltx4*>(smem) + (size_t)wt * WNF * WTF * WAVE + lane;
    auto give = [&](auto J0, auto J1) {
#pragma unroll
      for (int i = 0; i < WNF; ++i)
#pragma unroll
        for (int j = decltype(J0)::value; j < decltype(J1)::value; ++j)
          ex[(i * WTF + j) * WAVE] = eltx4{(elt)acc[i][j][0], (elt)acc[i][j][1], (elt)acc[i][j][2], (elt)acc[i][j][3]};
    };
    auto finish = [&](auto J0, auto J1, auto GATE) {
#pragma unroll
      for (int j = decltype(J0)::value; j < decltype(J1)::value; ++j) {
        const int t = t0 + (wt * WTF + j) * 16 + r16;
        if ((t >> 4) >= x_tt) continue;        // the token tile does not exist
#pragma unroll
        for (int i = 0; i < WNF; ++i) {
          const int c = n0 + i * 16 + gq * 4;
          if (c >= I) continue;
          const eltx4 other = ex[(i * WTF + j) * WAVE];
          eltx4 o = eltx4{0, 0, 0, 0};         // rows past T inside the last tile: zeros, as the separate kernel writes them
          if (t < T) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float own = (float)(elt)acc[i][j][r], oth = (float)other[r];
              o[r] = (elt)glu<OUT == OUT_CLIP ? MLORA_GLU_CLIPPED : MLORA_GLU_SILU>(decltype(GATE)::value ? own : oth, decltype(GATE)::value ? oth : own, ga);
            }
          }
          *reinterpret_cast<eltx4*>((elt*)yv + ((size_t)(c >> 5) * x_tt + (t >> 4)) * 512 + ((c & 31) >> 3) * 128 + (t & 15) * 8 + (c & 7)) = o;
        }
      }
    };
    typedef std::integral_constant<int, 0> Z;
    typedef std::integral_constant<int, H0> Hf;
    typedef std::integral_constant<int, WTF> W;
    if (wn == 0) give(Hf(), W());
    else give(Z(), Hf());
    __syncthreads();
    if (wn == 0) finish(Z(), Hf(), std::true_type());
    else finish(Hf(), W(), std::false_type());
    return;
  }
  if constexpr (OUT == OUT_F16) {
    // 16 tokens x (16 WNF) columns at a time through the wave's staging buffer: D[n][t] fragments in, token rows out
    elt* ostage = smem + wave * PP_OUT_ELEMS;
    constexpr int CPR = WNF * 2;               // 16-byte chunks per token row
#pragma unroll
    for (int j = 0; j < WTF; ++j) {
#pragma unroll
      for (int i = 0; i < WNF; ++i) {
        const f32x4 sacc = acc[i][j];
        *reinterpret_cast<eltx4*>(ostage + r16 * PP_OUT_LD + i * 16 + gq * 4) = eltx4{(elt)sacc[0], (elt)sacc[1], (elt)sacc[2], (elt)sacc[3]};
      }
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int q = 0; q < (16 * CPR + WAVE - 1) / WAVE; ++q) {
        const int c = q * 64 + lane;             // 16-byte chunk: token row c / CPR, columns (c % CPR) * 8 ..
        if ((16 * CPR) % WAVE != 0 && c >= 16 * CPR) break;
        const int tr = c / CPR, cc = (c % CPR) * 8;
        const int t = t0 + (wt * WTF + j) * 16 + tr;
        const int n = n0 + wn * WNF * 16 + cc;
        const eltx4 lo = *reinterpret_cast<const eltx4*>(ostage + tr * PP_OUT_LD + cc);
        const eltx4 hi = *reinterpret_cast<const eltx4*>(ostage + tr * PP_OUT_LD + cc + 4);
        if (t < T && n + 8 <= N) {
          st8((elt*)yv + (size_t)t * N + n, eltx8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
        } else if (t < T) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (n + e < N) ((elt*)yv)[(size_t)t * N + n + e] = lo[e];
            if (n + 4 + e < N) ((elt*)yv)[(size_t)t * N + n + 4 + e] = hi[e];
          }
        }
      }
      __builtin_amdgcn_wave_barrier();
    }
  } else {
#pragma unroll
    for (int j = 0; j < WTF; ++j) {
      const int t = t0 + (wt * WTF + j) * 16 + r16;
      if (t >= T) continue;
#pragma unroll
      for (int i = 0; i < WNF; ++i) {
        const int n = n0 + (wn * WNF + i) * 16 + gq * 4;
        if (n >= N) continue;
        const size_t o = (size_t)t * N + n;
        if constexpr (OUT == OUT_F32) {
          *reinterpret_cast<f32x4*>((float*)yv + o) = acc[i][j];
        } else {
          f32x4* p = reinterpret_cast<f32x4*>((float*)yv + o);
          *p = *p + acc[i][j];
        }
      }
    }
  }
}

// Block shape (16 ft tokens x 16 fn weight rows) and K slices of the mid-size kernel for a shape: the one that finishes first by
// two estimates, in units of 31 ns per 64-k stage.  A workgroup takes ft + 1.6 fn + 1 per stage - its operands through LDS, the
// products, the barrier (measured on 4096 x 12288: 0.46 us at 8 / 4, 0.63 at 8 / 8, 0.73 at 12 / 6, 0.92 at 16 / 8) - times the
// rounds that the compute units need for all workgroups.  All of them together take in their fragments, 0.0012 each, and those that
// miss the second-level caches: weights once, 0.02 each, tokens, 0.0107 each, once per XCD, or once per row block where these are fewer and the
// tokens more than 16 MiB (4568 tokens x 9984 x 400: seven row blocks of 64 99 us, five of 96 80).  The limit is a fit: over 200 sizes of 400 to
// 8192 tokens and 64 to 1040 rows the choice takes 0.6 % longer than the best of the nine on average and 14 % at most, with 32 MiB 0.8 and 17 %, without
// it 1.4 and 29 %.  The two overlap in part: root of the sum of squares.
// Measured where the choice matters, in us: 137 tokens, q/k/v 33.9 at 8 / 6, 36.0 at 12 / 4, 48 at 16 / 6; gate/up (22016 rows)
// 53.1 at 12 / 6, 60.8 at 16 / 6, 77.8 at 8 / 6; 300 tokens, q/k/v 49.8 at 12 / 6, 52.8 at 16 / 6, 71.5 at 8 / 8; o of 100 tokens in four
// slices 14.0 at 8 / 4, 17.1 at 8 / 8; 512 tokens x 4096 x 4096 29.6 at 8 / 4, 38.2 at 8 / 6.  Over 240 sizes the choice takes 1 % longer than the
// best of the nine on average, 10 % at most without and 29 % with K slices.
struct MidShape {
  int ft, fn, ksplit;
};
MidShape gemm_mid_shape(int T, int K, int N, int ksplit_max) {
  const int by_k = (K / 32) / 16 < 1 ? 1 : (K / 32) / 16;   // at least 16 k-steps per slice
  const int ks_cap = ksplit_max < by_k ? ksplit_max : by_k;
  int n_cu = gemm_n_cu();
  if (n_cu <= 0) n_cu = 256;
  MidShape best = {8, 4, 1};
  double least = 0;
  for (int ft = 8; ft <= 16; ft += 4)
    for (int fn = 4; fn <= 8; fn += 2) {
      const long rows = ceil_div(N, fn * 16), tb = ceil_div(T, ft * 16);
      long ks = n_cu / (rows * tb);
      ks = ks > ks_cap ? ks_cap : ks < 1 ? 1 : ks;
      const double rounds = (double)((rows * tb * ks + n_cu - 1) / n_cu), unit = ft + 1.6 * fn + 1;
      const double mine = rounds * unit / ks, tiles = ceil_div(T, 16);
      const int copies = (long)T * K * 2 > 16 << 20 && rows < 8 ? (int)rows : 8;       // of the tokens: one per XCD that has a row block
      const double all = 0.0012 * rows * (tiles + tb * fn) + 0.02 * ceil_div(N, 16) + 0.0107 * copies * tiles;
      const double cost = mine * mine + all * all;
      if (least == 0 || cost < least) {
        least = cost;
        best = MidShape{ft, fn, (int)ks};
      }
    }
  return best;
}

template <int OUT, int FT, int FN, bool GX = false, bool LORA = false>
int launch_gemm_mid_shape(void* y, float* part, int ld_part, int ksplit, const elt* xf, int x_tt, const elt* Wp, int T, int K, int N,
                          hipStream_t s, int gx_rows = 0, long gx_stride = 0, const GluArgs& ga = GluArgs(), const LinearDeltas& lo = LinearDeltas()) {
  constexpr size_t lds = (size_t)mid_stages(FT) * MID_KS * (FN + FT) * 512 * sizeof(elt);
  static_assert(lds >= (size_t)PP_WAVES * PP_OUT_ELEMS * sizeof(elt), "the output staging fits the ring");
  static const hipError_t configured =               // the attribute is per kernel, set once per process, by one thread
      hipFuncSetAttribute((const void*)gemm_mid_kernel<OUT, FT, FN, GX, LORA>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (configured != hipSuccess)
    return mlora_set_error(MLORA_ERR_LAUNCH, "linear_frag: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(configured));
  const dim3 grid(ceil_div(N, FN * 16), ksplit, ceil_div(T, FT * 16));       // (a gated product: ceil(I / (8 FN)) is the same)
  hipLaunchKernelGGL((gemm_mid_kernel<OUT, FT, FN, GX, LORA>), grid, dim3(PP_WAVES * WAVE), lds, s, y, part, ld_part, xf, x_tt, Wp, T, K, N, gx_rows, gx_stride, ga,
                     lo);
  return MLORA_OK;
}

template <int OUT, bool LORA = false>
int launch_gemm_mid(void* y, float* part, int ld_part, const MidShape& m, const elt* xf, int x_tt, const elt* Wp, int T, int K, int N,
                    hipStream_t s, const GluArgs& ga = GluArgs(), const LinearDeltas& lo = LinearDeltas()) {
#define MLORA_MID(FT, FN) \
  if (m.ft == FT && m.fn == FN) return launch_gemm_mid_shape<OUT, FT, FN, false, LORA>(y, part, ld_part, m.ksplit, xf, x_tt, Wp, T, K, N, s, 0, 0, ga, lo)
  MLORA_MID(8, 4);
  MLORA_MID(8, 6);
  MLORA_MID(8, 8);
  MLORA_MID(12, 4);
  MLORA_MID(12, 6);
  MLORA_MID(12, 8);
  MLORA_MID(16, 4);
  MLORA_MID(16, 6);
  MLORA_MID(16, 8);
#undef MLORA_MID
  return mlora_set_error(MLORA_ERR_UNSUPPORTED, "linear_frag: no block of %d x %d fragments", m.ft, m.fn);
}

template <int OUT, int FT, int FN, int WT_, int WN_>
int launch_gemm_lds(void* y, const elt* x, int ldx, const elt* Wp, int T, int K, int N, hipStream_t s) {
  constexpr size_t lds = 2 * (LBK / 32) * (FT + FN) * 512 * sizeof(elt);
  static const hipError_t configured =               // the attribute is per kernel, set once per process, by one thread
      lds > 64 * 1024 ? hipFuncSetAttribute((const void*)gemm_lds_kernel<OUT, FT, FN, WT_, WN_>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)
                      : hipSuccess;
  if (configured != hipSuccess)
    return mlora_set_error(MLORA_ERR_LAUNCH, "gemm_packed: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(configured));
  hipLaunchKernelGGL((gemm_lds_kernel<OUT, FT, FN, WT_, WN_>), dim3(ceil_div(N, FN * 16), ceil_div(T, FT * 16)), dim3(256), lds, s,
                     y, x, ldx, Wp, T, K, N);
  return MLORA_OK;
}

// Block shape by problem size.  256 tokens x 64 columns (wave 64 x 64) spread a few hundred tokens over all compute units, two blocks on
// each; a second round doubles their time, and from there on the persistent kernel is faster, up to half a round of whose blocks would be
// empty: 2500 tokens x 4096 x 4096 (640 small blocks) 102 us against 136, 700 x 4096 x 12288 (576) 101, 138, 3226 x 1024 x 2504 (520) 35, 42; 2425 x 512 x
// 3248 (510) 23, 20.  Not for a K that its blocks' ends outweigh: 281 x 64 x 23664 12.1, 9.2, 876 x 128 x 9648 13.6, 11.8, 1410 x 256 x 6520 15.9, 16.6.
template <int OUT>
int launch_gemm_lds_auto(void* y, const elt* x, int ldx, const elt* Wp, int T, int K, int N, hipStream_t s) {
  const long nb = (long)ceil_div(T, 256) * ceil_div(N, 256), cu = gemm_n_cu() > 0 ? gemm_n_cu() : 256;
  const bool large = nb >= cu, second = (long)ceil_div(T, 256) * ceil_div(N, 64) > 2 * cu && K >= 256;
  // x rows must be 16-byte aligned for the direct-to-LDS loads (ldx % 8 == 0 is checked; the base may be a slice)
  if ((large || second) && ((uintptr_t)x & 15) == 0 && K % 64 == 0) return launch_gemm_pp<OUT>(y, x, ldx, 0, Wp, T, K, N, s);
  if (large) return launch_gemm_lds<OUT, 16, 16, 8, 8>(y, x, ldx, Wp, T, K, N, s);
  return launch_gemm_lds<OUT, 16, 4, 4, 4>(y, x, ldx, Wp, T, K, N, s);
}

template <bool PACKED>
int gemm_dispatch(const char* who, void* y, int y_dtype, int mode, const void* x, int ldx, const void* W, int T, int K,
                  int N, void* stream) {
  if (int e = mlora_check_linear(who, y, y_dtype, mode, x, ldx, W, T, K, N)) return e;
  if (T == 0) return MLORA_OK;
  MLORA_CHECK(ceil_div(T, 128) <= 65535, MLORA_ERR_UNSUPPORTED, "%s: T=%d too large", who, T);
  const dim3 grid(ceil_div(N, 128), ceil_div(T, 128)), block(256);
  hipStream_t s = (hipStream_t)stream;
  const elt* xp = (const elt*)x;
  const elt* Wp = (const elt*)W;
  if constexpr (PACKED) {
    if (T > 128) {
      int e;
      if (mode == MLORA_ACCUMULATE) e = launch_gemm_lds_auto<OUT_ACC_F32>(y, xp, ldx, Wp, T, K, N, s);
      else if (y_dtype == MLORA_F32) e = launch_gemm_lds_auto<OUT_F32>(y, xp, ldx, Wp, T, K, N, s);
      else e = launch_gemm_lds_auto<OUT_F16>(y, xp, ldx, Wp, T, K, N, s);
      return e ? e : mlora_launch_status(who);
    }
  }
  if (mode == MLORA_ACCUMULATE) hipLaunchKernelGGL((gemm_kernel<OUT_ACC_F32, PACKED>), grid, block, 0, s, y, xp, ldx, Wp, T, K, N);
  else if (y_dtype == MLORA_F32) hipLaunchKernelGGL((gemm_kernel<OUT_F32, PACKED>), grid, block, 0, s, y, xp, ldx, Wp, T, K, N);
  else hipLaunchKernelGGL((gemm_kernel<OUT_F16, PACKED>), grid, block, 0, s, y, xp, ldx, Wp, T, K, N);
  return mlora_launch_status(who);
}

}  // namespace

extern "C" int mlora_gemm(void* y, int y_dtype, int mode, const void* x, int ldx, const void* W, int T, int K, int N,
                          void* stream) {
  return gemm_dispatch<false>("gemm", y, y_dtype, mode, x, ldx, W, T, K, N, stream);
}

extern "C" int mlora_gemm_packed(void* y, int y_dtype, int mode, const void* x, int ldx, const void* Wp, int T, int K,
                                 int N, void* stream) {
  return gemm_dispatch<true>("gemm_packed", y, y_dtype, mode, x, ldx, Wp, T, K, N, stream);
}

extern "C" int mlora_linear(void* y, int y_dtype, int mode, const void* x, int ldx, const void* W, int T, int K, int N,
                            void* stream) {
  if (T <= 64) return mlora_gemv(y, y_dtype, mode, x, ldx, W, T, K, N, stream);
  return mlora_gemm(y, y_dtype, mode, x, ldx, W, T, K, N, stream);
}

extern "C" int mlora_linear_packed(void* y, int y_dtype, int mode, const void* x, int ldx, const void* Wp, int T, int K,
                                   int N, void* stream) {
  if (T <= 64) return mlora_gemv_packed(y, y_dtype, mode, x, ldx, Wp, T, K, N, stream);
  return mlora_gemm_packed(y, y_dtype, mode, x, ldx, Wp, T, K, N, stream);
}

extern "C" int mlora_gemv_frag(void* y, int y_dtype, int mode, const void* xf, const void* Wp, int T, int K, int N, void* stream);

// 256 x 256 output blocks: enough of them to give every compute unit one (the forms with an epilogue of their own - a gated product, LoRA deltas -
// take it from there on).  K in whole 64, here and wherever the persistent kernel is chosen: its ring walks single steps of 32 k, but an odd number of them
// has been neither tested nor measured.  256 is the number of compute units; the plain linear and the gated product take the kernel from half of
// that on (persistent_pays), LoRA stages have not been measured there.  Just above one round the plain linear goes back to the mid-size kernel, by an eighth of a
// round; the gated product and the LoRA stages stay, they have not been compared there.
extern "C" int mlora_gemm_frag_preferred(int T, int K, int N) {
  return T > 64 && K > 0 && K % 64 == 0 && N > 0 && (long)ceil_div(T, PP_F * 16) * ceil_div(N, PP_F * 16) >= 256;
}

// The plain linear: the persistent kernel or the mid-size one.  The first takes whole rounds of one 256 x 256 block per compute unit: padding
// and empty units cost as much as products.  So what is asked is T N / 2^16, the blocks' worth of products.  In one round more than half of
// the chip: up to there the mid-size kernel has a round of its own largest blocks, of half that size.  Above one round what pays for the second:
// a whole first one and an eighth, less for small K, where the mid-size kernel's block ends weigh more - but not where results are added to fp32, since both
// kernels' ends then wait for memory.
// Measured, persistent / mid-size, us.  One round: 113 (1843 x 2304 x 4032) 46 / 37, 120 (640 x 4096 x 12288) 77 / 72, 126 (1500 x 1024 x 5504) 26 / 29,
// 128 (2048 x 4096 x 4096) 77 / 63, 129 (1500 x 2048 x 5632) 41 / 47, 134 (400 x 4096 x 22016) 81 / 107, 141 (3000 x 2048 x 3072) 45 / 45, 144 (768 x 4096 x 12288)
// 78 / 86, 156 (2500 x 4096 x 4096) 78 / 93, 172 (512 x 4096 x 22016) 82 / 112.  Two, K from 1280 on: 190 (548 x 3264 x 22704) 122 / 105, 258 (3000 x 2048 x 5632)
// 82 / 76, 258 (768 x 4096 x 22016) 152 / 152, 281 (1500 x 4096 x 12288) 155 / 147, 302 (900 x 4096 x 22016) 161 / 183, 394 (900 x 4096 x 28672) 173 / 231; below:
// 235 (3123 x 1024 x 4928) 46 / 43, 251 (1515 x 1024 x 10864) 46 / 44, 252 (2549 x 256 x 6504) 21 / 21, 274 (815 x 384 x 22032) 26 / 35, 290 (643 x 320 x 29560)
// 24 / 32.  Added to: 262 (2281 x 64 x 7520) 39 / 30, 272 (904 x 384 x 19904) 50 / 50, 277 (1268 x 512 x 14296) 55 / 52, 288 (3072 x 2752 x 6136) 134 / 123, 297
// (3725 x 384 x 5224) 50 / 54, 298 (1451 x 1024 x 13464) 75 / 78, 301 (1492 x 192 x 13216) 44 / 40, 317 (1515 x 2048 x 13720) 115 / 118.  Over 280 sizes of
// 60 to 560 blocks the choice takes 1.3 % longer than the better one on average, 33 % at most (247 x 256 x 33752, just below half a round, 12 / 17).  Up to
// 128 tokens half of its work is padding.
static bool persistent_pays(int T, int K, int N, bool accumulate) {
  const long cu = gemm_n_cu() > 0 ? gemm_n_cu() : 256, nb = (long)ceil_div(T, PP_F * 16) * ceil_div(N, PP_F * 16);
  if (K % 64 || T <= 128) return false;
  const long block = PP_F * 16 * PP_F * 16;
  return nb <= cu ? (long)T * N * 2 > cu * block : (long)T * N * 32 >= cu * (accumulate ? 37 : K >= 1280 ? 36 : 32) * block;
}

extern "C" int mlora_linear_frag(void* y, int y_dtype, int mode, const void* xf, const void* Wp, int T, int K, int N,
                                 void* stream) {
  if (T <= 64) return mlora_gemv_frag(y, y_dtype, mode, xf, Wp, T, K, N, stream);
  if (int e = mlora_check_linear("linear_frag", y, y_dtype, mode, xf, K, Wp, T, K, N)) return e;
  MLORA_CHECK(K % 32 == 0, MLORA_ERR_UNSUPPORTED, "linear_frag: K %% 32 != 0 (K=%d)", K);
  MLORA_CHECK(((uintptr_t)xf & 15) == 0, MLORA_ERR_INVALID, "linear_frag: xf must be 16-byte aligned");
  hipStream_t s = (hipStream_t)stream;
  const elt* x = (const elt*)xf;
  const elt* W = (const elt*)Wp;
  const int tt = mlora_frag_tiles(T);
  int e;
  if (persistent_pays(T, K, N, mode == MLORA_ACCUMULATE)) {
    if (mode == MLORA_ACCUMULATE) e = launch_gemm_pp<OUT_ACC_F32>(y, x, 0, tt, W, T, K, N, s);
    else if (y_dtype == MLORA_F32) e = launch_gemm_pp<OUT_F32>(y, x, 0, tt, W, T, K, N, s);
    else e = launch_gemm_pp<OUT_F16>(y, x, 0, tt, W, T, K, N, s);
  } else {
    const MidShape m = gemm_mid_shape(T, K, N, 1);
    if (mode == MLORA_ACCUMULATE) e = launch_gemm_mid<OUT_ACC_F32>(y, nullptr, 0, m, x, tt, W, T, K, N, s);
    else if (y_dtype == MLORA_F32) e = launch_gemm_mid<OUT_F32>(y, nullptr, 0, m, x, tt, W, T, K, N, s);
    else e = launch_gemm_mid<OUT_F16>(y, nullptr, 0, m, x, tt, W, T, K, N, s);
  }
  return e ? e : mlora_launch_status("linear_frag");
}

extern "C" int mlora_linear_frag_clipglu(void* act, const void* xf, const void* Wp, int T, int K, int I, float scale, float limit,
                                         float alpha, void* stream) {
  MLORA_CHECK(act && xf && Wp, MLORA_ERR_INVALID, "linear_frag_clipglu: null pointer");
  MLORA_CHECK(T > 0 && K > 0 && I > 0 && I % 32 == 0 && I <= (1 << 29), MLORA_ERR_UNSUPPORTED,
              "linear_frag_clipglu: need I %% 32 == 0 (T=%d K=%d I=%d)", T, K, I);
  MLORA_CHECK(mlora_gemm_frag_preferred(T, K, 2 * I) && (((uintptr_t)xf | (uintptr_t)act) & 15) == 0, MLORA_ERR_UNSUPPORTED,
              "linear_frag_clipglu: only shapes of the persistent GEMM (mlora_gemm_frag_preferred; T=%d K=%d N=%d)", T, K, 2 * I);
  return mlora_linear_frag_glu(act, xf, Wp, T, K, I, MLORA_GLU_CLIPPED, scale, limit, alpha, stream);
}

// act = the gated product of [gate | up] = xf . Wp^T for more than 64 tokens: on the persistent kernel where mlora_gemm_frag_preferred or the plain linear takes it
// (which differ just above one round of its blocks), else on the mid-size one.  The clipped product is of unrounded sums on the first, of rounded ones on the second.  A product
// behind the linear writes and reads T x 2 I elements once more and costs a launch (a floor of 2.5 us); what is left in its place is the exchange
// of half a block through LDS.  Linear and product behind it -> here, in a row of launches (K, I): 512, 1376 at 65 / 512 / 1024 tokens 7.6 / 9.9 /
// 13.3 -> 6.3 / 6.7 / 8.9 us; 2048, 5632: 14.7 / 34.8 / 52.3 -> 13.1 / 31.3 / 49.3; 2880, 2880: 17.4 / 28.6 / 42.7 -> 15.9 / 25.1 / 39.8; 4096,
// 11008 at 65 / 512: 31.6 / 87.7 -> 30.0 / 82.9 (weights from HBM each time).  Never slower on the mid-size kernel, so there is no rule.
extern "C" int mlora_linear_frag_glu(void* act, const void* xf, const void* Wp, int T, int K, int I, int kind, float scale, float limit, float alpha,
                                     void* stream) {
  MLORA_CHECK(act && xf && Wp, MLORA_ERR_INVALID, "linear_frag_glu: null pointer");
  MLORA_CHECK(kind == MLORA_GLU_SILU || kind == MLORA_GLU_CLIPPED, MLORA_ERR_INVALID, "linear_frag_glu: bad kind %d", kind);
  MLORA_CHECK(T > 64 && K > 0 && K % 32 == 0 && I > 0 && I % 32 == 0 && I <= (1 << 29) && (((uintptr_t)xf | (uintptr_t)act) & 15) == 0,
              MLORA_ERR_UNSUPPORTED, "linear_frag_glu: more than 64 tokens, K and I in whole 32, aligned operands (T=%d K=%d I=%d)", T, K, I);
  const GluArgs ga{scale, limit, alpha};
  const elt *x = (const elt*)xf, *W = (const elt*)Wp;
  const int tt = mlora_frag_tiles(T);
  hipStream_t s = (hipStream_t)stream;
  int e;
  if (mlora_gemm_frag_preferred(T, K, 2 * I) || persistent_pays(T, K, 2 * I, false)) {
    e = kind == MLORA_GLU_SILU ? launch_gemm_pp<OUT_SILU>(act, x, 0, tt, W, T, K, 2 * I, s) : launch_gemm_pp<OUT_CLIP>(act, x, 0, tt, W, T, K, 2 * I, s, PPLora(), ga);
  } else {
    MLORA_CHECK(ceil_div(T, 128) <= 65535, MLORA_ERR_UNSUPPORTED, "linear_frag_glu: T=%d too large", T);
    const MidShape m = gemm_mid_shape(T, K, 2 * I, 1);
    e = kind == MLORA_GLU_SILU ? launch_gemm_mid<OUT_SILU>(act, nullptr, 0, m, x, tt, W, T, K, 2 * I, s) : launch_gemm_mid<OUT_CLIP>(act, nullptr, 0, m, x, tt, W, T, K, 2 * I, s, ga);
  }
  return e ? e : mlora_launch_status("linear_frag_glu");
}

#ifndef MLORA_ELT_BF16      // the adapter kernels are fp16
// Whether the linears with deltas below serve a shape: where neither the plain one nor the gated product takes the persistent kernel.
static bool mid_deltas_serve(int T, int K, int N, bool accumulate) {
  return T > 64 && ceil_div(T, 128) <= 65535 && K >= 32 && K % 32 == 0 && !mlora_gemm_frag_preferred(T, K, N) && !persistent_pays(T, K, N, accumulate);
}

// What the deltas cost in there is a round trip to memory per 32 ranks and adapter (up to 64 tokens: per tile of 16, and shared by eight waves); on their own they are a launch that reads and
// writes y.  Passes of two layers, us, on their own / in the linear, by rounds: 1 (7B, q, k, v and o, rank 16, 80 tokens) 423 / 404, (600 tokens) 1066 /
// 1012, (hidden 1024, all seven, 200 tokens) 314 / 285; 2 (7B, all, rank 64, 300 tokens) 915 / 829; 3 (rank 16, 8 x 60 tokens, q, k, v, o) 774 / 737; 6
// (rank 64, 4 x 90, all) 1022 / 1004; 7 (rank 16, 8 x 60) 778 / 752; 14 (rank 64, 8 x 50, all) 1002 / 1010, (hidden 1024, 8 x 150) 548 / 559.
// Decode steps: (7B, rank 32, 2 requests, all) 407 / 371; (rank 64, one, all) 385 / 340, (hidden 1024) 197 / 145; (rank 32, 16) 340 / 331.  The line is one tile
// of tokens, whatever they name (a step's bits must not follow its ids): of more tiles (rank 16, 64 of one adapter, q, k, v, o) 408 / 408, (hidden 1024, rank
// 32, 40) 268 / 280, (rank 64, 32 of seven) 401 / 411, (rank 64, 49 of three) 441 / 460.
extern "C" int mlora_linear_frag_deltas_pay(int T, int K, int N, int accumulate, int r, int n_distinct) {
  const long rounds = (long)ceil_div(r, 32) * n_distinct;
  if (T <= 64) return T > 0 && T <= 16 && K > 0 && K % 32 == 0 && N % 16 == 0 && rounds > 0;
  return mid_deltas_serve(T, K, N, accumulate != 0) && rounds > 0 && rounds <= 8;
}

// the shrink of the projections into the workspace (gather_mm.hip), and what the kernel above reads of it
int mlora_lora_shrink_ranges(const void* const* A, int n_proj, const void* xf, const int32_t* tok_adapter, int T, int K, int r, int n_ad, float* v, int most,
                             void* stream);
int mlora_gemv_deltas(void* y, int y_dtype, int mode, float* part, int ks, const void* xf, const void* Wp, int T, int K, int N, const LinearDeltas& ld, void* stream);
static int mid_lora(const char* who, LinearDeltas& lo, const mlora_lora_bucket* projs, int n_proj, const int32_t* n_begin, const int32_t* n_rows, const void* xf,
                    const int32_t* ids, int T, int K, int N, void* workspace, size_t workspace_bytes, void* stream) {
  MLORA_CHECK(projs && n_begin && n_rows && ids && n_proj >= 1 && n_proj <= 3, MLORA_ERR_INVALID, "%s: null pointer or n_proj=%d outside 1..3", who, n_proj);
  const int r = projs[0].r, n_ad = projs[0].n_ad;
  MLORA_CHECK((r == 8 || r == 16 || r == 32 || r == 64) && n_ad > 0 && n_ad <= 65535, MLORA_ERR_UNSUPPORTED, "%s: rank %d not in {8, 16, 32, 64} or bad n_ad %d",
              who, r, n_ad);
  const size_t need = (size_t)n_proj * mlora_gather_mm_workspace_bytes(T, K, r);
  MLORA_CHECK(workspace && workspace_bytes >= need && ((uintptr_t)workspace & 15) == 0, MLORA_ERR_WORKSPACE, "%s: workspace of %zu bytes given, %zu needed (16-byte aligned)",
              who, workspace_bytes, need);
  const void* A[3];
  for (int i = 0; i < n_proj; ++i) {
    const mlora_lora_bucket& p = projs[i];
    MLORA_CHECK(p.A && p.B, MLORA_ERR_INVALID, "%s: null table of projection %d", who, i);
    MLORA_CHECK(p.r == r && p.n_ad == n_ad && p.scaling == projs[0].scaling, MLORA_ERR_UNSUPPORTED, "%s: projections of different ranks, adapters or scalings", who);
    MLORA_CHECK(n_begin[i] >= 0 && n_rows[i] > 0 && n_begin[i] <= N - n_rows[i], MLORA_ERR_UNSUPPORTED, "%s: rows %d..%d of projection %d of %d rows", who,
                n_begin[i], n_begin[i] + n_rows[i], i, N);
    A[i] = p.A;
    lo.B[i] = (const elt*)p.B; lo.n_begin[i] = n_begin[i]; lo.n_rows[i] = n_rows[i];
  }
  lo.v = (const float*)workspace; lo.ids = ids; lo.scaling = projs[0].scaling;
  lo.n_proj = n_proj; lo.r = r; lo.n_ad = n_ad;
  // (a long K up to 64 tokens: twice the ranges, so that the sums are as exact as elsewhere; a second round of loads, 1 us)
  lo.ranges = mlora_lora_shrink_ranges(A, n_proj, xf, ids, T, K, r, n_ad, (float*)workspace, T <= 64 && K > 8192 ? 2 * DELTA_RANGES : DELTA_RANGES, stream);
  return MLORA_OK;
}

extern "C" int mlora_linear_frag_deltas(void* y, int y_dtype, int mode, float* part, int ks, const void* xf, const void* Wp, int T, int K, int N,
                                        const mlora_lora_bucket* projs, int n_proj, const int32_t* n_begin, const int32_t* n_rows,
                                        const int32_t* tok_adapter, void* workspace, size_t workspace_bytes, void* stream) {
  if (int e = mlora_check_linear("linear_frag_deltas", y, y_dtype, mode, xf, K, Wp, T, K, N)) return e;
  MLORA_CHECK((T <= 64 ? T > 0 && K % 32 == 0 && N % 16 == 0 : mid_deltas_serve(T, K, N, mode == MLORA_ACCUMULATE)) && ((uintptr_t)xf & 15) == 0,
              MLORA_ERR_UNSUPPORTED, "linear_frag_deltas: up to 64 tokens, or shapes of the mid-size kernel (mlora_linear_frag_deltas_pay; T=%d K=%d N=%d)", T, K, N);
  MLORA_CHECK(ks == 1 || (ks > 1 && ks <= 4 && part && mode == MLORA_ACCUMULATE && K / 32 / ks >= (T <= 64 ? 8 : 1)), MLORA_ERR_INVALID,
              "linear_frag_deltas: ks=%d slices (accumulating only), or no partials buffer", ks);
  LinearDeltas lo = {};
  if (int e = mid_lora("linear_frag_deltas", lo, projs, n_proj, n_begin, n_rows, xf, tok_adapter, T, K, N, workspace, workspace_bytes, stream)) return e;
  if (T <= 64) return mlora_gemv_deltas(y, y_dtype, mode, part, ks, xf, Wp, T, K, N, lo, stream);
  hipStream_t s = (hipStream_t)stream;
  MidShape m = gemm_mid_shape(T, K, N, ks);
  m.ksplit = ks;                               // the caller's partial buffers were sized for ks slices
  const elt *x = (const elt*)xf, *W = (const elt*)Wp;
  const int tt = mlora_frag_tiles(T);
  int e;
  if (mode == MLORA_ACCUMULATE) e = launch_gemm_mid<OUT_ACC_F32, true>(y, part, N, m, x, tt, W, T, K, N, s, GluArgs(), lo);
  else if (y_dtype == MLORA_F32) e = launch_gemm_mid<OUT_F32, true>(y, nullptr, 0, m, x, tt, W, T, K, N, s, GluArgs(), lo);
  else e = launch_gemm_mid<OUT_F16, true>(y, nullptr, 0, m, x, tt, W, T, K, N, s, GluArgs(), lo);
  return e ? e : mlora_launch_status("linear_frag_deltas");
}

int mlora_gemv_silu_deltas(void* act, const void* xf, const void* Wil_p, int T, int K, int I, const LinearDeltas& ld, void* stream);
extern "C" int mlora_gemv_frag_silu_deltas(void* act, const void* xf, const void* Wil_p, int T, int K, int I, const mlora_lora_bucket* projs, int n_proj,
                                           const int32_t* n_begin, const int32_t* n_rows, const int32_t* tok_adapter, void* workspace,
                                           size_t workspace_bytes, void* stream) {
  MLORA_CHECK(act && xf && Wil_p, MLORA_ERR_INVALID, "gemv_frag_silu_deltas: null pointer");
  MLORA_CHECK(T > 0 && T <= 64 && K > 0 && K % 32 == 0 && I > 0 && I % 32 == 0 && I <= (1 << 29) && (((uintptr_t)xf | (uintptr_t)act) & 15) == 0,
              MLORA_ERR_UNSUPPORTED, "gemv_frag_silu_deltas: up to 64 tokens, K and I in whole 32, aligned operands (T=%d K=%d I=%d)", T, K, I);
  LinearDeltas lo = {};
  if (int e = mid_lora("gemv_frag_silu_deltas", lo, projs, n_proj, n_begin, n_rows, xf, tok_adapter, T, K, 2 * I, workspace, workspace_bytes, stream)) return e;
  return mlora_gemv_silu_deltas(act, xf, Wil_p, T, K, I, lo, stream);
}

extern "C" int mlora_linear_frag_silu_deltas(void* act, const void* xf, const void* Wp, int T, int K, int I, const mlora_lora_bucket* projs, int n_proj,
                                             const int32_t* n_begin, const int32_t* n_rows, const int32_t* tok_adapter, void* workspace,
                                             size_t workspace_bytes, void* stream) {
  MLORA_CHECK(act && xf && Wp, MLORA_ERR_INVALID, "linear_frag_silu_deltas: null pointer");
  MLORA_CHECK(I > 0 && I % 32 == 0 && I <= (1 << 29) && mid_deltas_serve(T, K, 2 * I, false) && (((uintptr_t)xf | (uintptr_t)act) & 15) == 0,
              MLORA_ERR_UNSUPPORTED, "linear_frag_silu_deltas: only shapes of the mid-size kernel, I in whole 32 (T=%d K=%d I=%d)", T, K, I);
  LinearDeltas lo = {};
  if (int e = mid_lora("linear_frag_silu_deltas", lo, projs, n_proj, n_begin, n_rows, xf, tok_adapter, T, K, 2 * I, workspace, workspace_bytes, stream)) return e;
  const int e = launch_gemm_mid<OUT_SILU, true>(act, nullptr, 0, gemm_mid_shape(T, K, 2 * I, 1), (const elt*)xf, mlora_frag_tiles(T), (const elt*)Wp, T, K, 2 * I,
                                                (hipStream_t)stream, GluArgs(), lo);
  return e ? e : mlora_launch_status("linear_frag_silu_deltas");
}

extern "C" int mlora_linear_frag_lora(void* y, int y_dtype, int mode, const void* xf, const void* Wp, int T, int K, int N,
                                      const mlora_fused_lora* projs, int n_proj, const int32_t* blk_adapter, int r, void* stream) {
  if (int e = mlora_check_linear("linear_frag_lora", y, y_dtype, mode, xf, K, Wp, T, K, N)) return e;
  MLORA_CHECK(mlora_gemm_frag_preferred(T, K, N) && ((uintptr_t)xf & 15) == 0, MLORA_ERR_UNSUPPORTED,
              "linear_frag_lora: only shapes of the persistent GEMM (mlora_gemm_frag_preferred; T=%d K=%d N=%d)", T, K, N);
  MLORA_CHECK(projs && blk_adapter && n_proj >= 1 && n_proj <= 3 && (r == 32 || r == 64), MLORA_ERR_UNSUPPORTED,
              "linear_frag_lora: 1..3 projections of rank 32 or 64 (n_proj=%d r=%d)", n_proj, r);
  PPLora lo = {};
  for (int i = 0; i < n_proj; ++i) {
    const mlora_fused_lora& p = projs[i];
    MLORA_CHECK(p.B && p.v_hi && p.v_lo && (((uintptr_t)p.B | (uintptr_t)p.v_hi | (uintptr_t)p.v_lo) & 15) == 0, MLORA_ERR_INVALID,
                "linear_frag_lora: null or unaligned table of projection %d", i);
    // a 256-row block of the GEMM must lie inside one projection
    MLORA_CHECK(p.n_begin >= 0 && p.n_rows > 0 && p.n_begin % (PP_F * 16) == 0 && p.n_begin + p.n_rows <= N &&
                    (p.n_rows % (PP_F * 16) == 0 || p.n_begin + p.n_rows == N),
                MLORA_ERR_UNSUPPORTED, "linear_frag_lora: rows %d..%d of projection %d do not fall on 256-row blocks", p.n_begin,
                p.n_begin + p.n_rows, i);
    lo.B[i] = (const elt*)p.B; lo.vh[i] = (const elt*)p.v_hi; lo.vl[i] = (const elt*)p.v_lo;
    lo.n_begin[i] = p.n_begin; lo.n_rows[i] = p.n_rows;
  }
  lo.n_proj = n_proj; lo.r = r; lo.blk_adapter = blk_adapter;
  hipStream_t s = (hipStream_t)stream;
  const int tt = mlora_frag_tiles(T);
  int e;
  if (mode == MLORA_ACCUMULATE) e = launch_gemm_pp<OUT_ACC_F32>(y, (const elt*)xf, 0, tt, (const elt*)Wp, T, K, N, s, lo);
  else if (y_dtype == MLORA_F32) e = launch_gemm_pp<OUT_F32>(y, (const elt*)xf, 0, tt, (const elt*)Wp, T, K, N, s, lo);
  else e = launch_gemm_pp<OUT_F16>(y, (const elt*)xf, 0, tt, (const elt*)Wp, T, K, N, s, lo);
  return e ? e : mlora_launch_status("linear_frag_lora");
}
#endif

extern "C" int mlora_linear_frag_silu(void* act, const void* xf, const void* Wp, int T, int K, int I, const mlora_fused_lora* projs,
                                      int n_proj, const int32_t* blk_adapter, int r, void* stream) {
  MLORA_CHECK(act && xf && Wp, MLORA_ERR_INVALID, "linear_frag_silu: null pointer");
  MLORA_CHECK(T > 0 && K > 0 && I > 0 && I % 32 == 0 && I <= (1 << 29), MLORA_ERR_UNSUPPORTED,
              "linear_frag_silu: need I %% 32 == 0 (T=%d K=%d I=%d)", T, K, I);
  MLORA_CHECK(mlora_gemm_frag_preferred(T, K, 2 * I) && (((uintptr_t)xf | (uintptr_t)act) & 15) == 0, MLORA_ERR_UNSUPPORTED,
              "linear_frag_silu: only shapes of the persistent GEMM (mlora_gemm_frag_preferred; T=%d K=%d N=%d)", T, K, 2 * I);
  MLORA_CHECK(n_proj >= 0 && n_proj <= 2, MLORA_ERR_UNSUPPORTED, "linear_frag_silu: at most the gate and the up projection (n_proj=%d)", n_proj);
  PPLora lo = {};
  if (n_proj > 0) {
    MLORA_CHECK(projs && blk_adapter && (r == 32 || r == 64), MLORA_ERR_UNSUPPORTED,
                "linear_frag_silu: projections of rank 32 or 64 with the blocks' adapters (r=%d)", r);
    for (int i = 0; i < n_proj; ++i) {
      const mlora_fused_lora& p = projs[i];
      MLORA_CHECK(p.B && p.v_hi && p.v_lo && (((uintptr_t)p.B | (uintptr_t)p.v_hi | (uintptr_t)p.v_lo) & 15) == 0, MLORA_ERR_INVALID,
                  "linear_frag_silu: null or unaligned table of projection %d", i);
      MLORA_CHECK((p.n_begin == 0 || p.n_begin == I) && p.n_rows == I, MLORA_ERR_UNSUPPORTED,
                  "linear_frag_silu: projection %d must be the gate rows 0..I or the up rows I..2I (n_begin=%d n_rows=%d I=%d)", i,
                  p.n_begin, p.n_rows, I);
      const int slot = p.n_begin == 0 ? 0 : 1;
      MLORA_CHECK(lo.B[slot] == nullptr, MLORA_ERR_INVALID, "linear_frag_silu: two projections over the same rows");
      lo.B[slot] = (const elt*)p.B; lo.vh[slot] = (const elt*)p.v_hi; lo.vl[slot] = (const elt*)p.v_lo;
      lo.n_begin[slot] = p.n_begin; lo.n_rows[slot] = p.n_rows;
    }
    lo.n_proj = n_proj; lo.r = r; lo.blk_adapter = blk_adapter;
  }
  const int e = launch_gemm_pp<OUT_SILU>(act, (const elt*)xf, 0, mlora_frag_tiles(T), (const elt*)Wp, T, K, 2 * I, (hipStream_t)stream, lo);
  return e ? e : mlora_launch_status("linear_frag_silu");
}

#ifdef MLORA_ELT_BF16
// One expert linear over a plan of 256-place tiles: xf places in fragment order (x_tt tiles of 16), y as PPGroup says.
template <int OUT>
static int launch_gemm_grouped(void* y, const elt* xf, int x_tt, const elt* Wp, int K, int N, int max_tiles, const PPGroup& gr, hipStream_t s) {
  constexpr size_t lds = ((size_t)PP_STAGES * PP_STAGE_ELEMS + (size_t)PP_WAVES * PP_OUT_ELEMS) * sizeof(elt);
  static const hipError_t configured =
      hipFuncSetAttribute((const void*)gemm_pp_kernel<OUT, false, true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (configured != hipSuccess)
    return mlora_set_error(MLORA_ERR_LAUNCH, "moe_linear: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(configured));
  const int gx = OUT == OUT_SILU ? ceil_div(N / 2, PP_F * 8) : ceil_div(N, PP_F * 16);
  int n_cu = gemm_n_cu();
  if (n_cu <= 0) n_cu = 256;
  const long nb = (long)gx * max_tiles;
  hipLaunchKernelGGL((gemm_pp_kernel<OUT, false, true>), dim3(nb < n_cu ? (int)nb : n_cu), dim3(PP_WAVES * WAVE), lds, s, y, xf, 0, x_tt, Wp,
                     x_tt * 16, K, N, gx, max_tiles, PPLora(), GluArgs(), gr);
  return MLORA_OK;
}

int mlora_gemm_grouped(void* y, const void* xf, int x_tt, const void* Wp, const MoePlan& plan, int max_tiles, int K, int N, int act, float alpha,
                       void* stream) {
  MLORA_CHECK(K % 64 == 0 && N % 32 == 0 && x_tt > 0 && max_tiles > 0, MLORA_ERR_UNSUPPORTED, "moe_linear: K=%d N=%d", K, N);   // the caller's checks say more
  PPGroup gr;
  gr.plan = plan;
  gr.w_elems = (size_t)N * K * (act == MLORA_ACT_GLU ? 2 : 1);
  gr.alpha = alpha;
  hipStream_t s = (hipStream_t)stream;
  const int e = act == MLORA_ACT_GLU ? launch_gemm_grouped<OUT_SILU>(y, (const elt*)xf, x_tt, (const elt*)Wp, K, 2 * N, max_tiles, gr, s)
                : act == MLORA_ACT_RELU2 ? launch_gemm_grouped<OUT_RELU2>(y, (const elt*)xf, x_tt, (const elt*)Wp, K, N, max_tiles, gr, s)
                                         : launch_gemm_grouped<OUT_F16>(y, (const elt*)xf, x_tt, (const elt*)Wp, K, N, max_tiles, gr, s);
  return e ? e : mlora_launch_status("moe_linear");
}
#endif

#ifdef MLORA_ELT_BF16
extern "C" int mlora_gemm_frag_groups(void* y, const void* xf, long x_stride, int group_rows, const void* Wp, int T, int K, int N, void* stream) {
  if (int e = mlora_check_linear("gemm_frag_groups", y, MLORA_F16, MLORA_STORE, xf, K, Wp, T, K, N)) return e;
  MLORA_CHECK(T > 64 && T <= 65535 && group_rows > 0 && group_rows % 64 == 0 && N % group_rows == 0 && x_stride % 8 == 0 && ((uintptr_t)xf & 15) == 0,
              MLORA_ERR_UNSUPPORTED, "gemm_frag_groups: more than 64 tokens and groups of whole 64 rows (T=%d rows=%d N=%d)", T, group_rows, N);
  hipStream_t s = (hipStream_t)stream;
  const elt* x = (const elt*)xf;
  const elt* W = (const elt*)Wp;
  const int tt = mlora_frag_tiles(T);
  int e;
  if (group_rows % 128 == 0 && (long)(N / 64) * ceil_div(T, 128) > 256)        // 128 rows a workgroup where that leaves one for every unit
    e = T <= 128 ? launch_gemm_mid_shape<OUT_F16, 8, 8, true>(y, nullptr, 0, 1, x, tt, W, T, K, N, s, group_rows, x_stride)
                 : launch_gemm_mid_shape<OUT_F16, 16, 8, true>(y, nullptr, 0, 1, x, tt, W, T, K, N, s, group_rows, x_stride);
  else
    e = launch_gemm_mid_shape<OUT_F16, 8, 4, true>(y, nullptr, 0, 1, x, tt, W, T, K, N, s, group_rows, x_stride);
  return e ? e : mlora_launch_status("gemm_frag_groups");
}

int mlora_gemv_ksplit_store(float* y, float* part, int ks, const void* xf, const void* Wp, int T, int K, int N, void* stream);

// y [T, N] fp32 = xf . Wp^T over ks K slices (mlora_gemv_ksplit): slice 0 into y, slices 1.. into part[ks - 1][T][N]
extern "C" int mlora_linear_ksplit_store(float* y, float* part, int ks, const void* xf, const void* Wp, int T, int K, int N, void* stream) {
  if (int e = mlora_check_linear("linear_ksplit_store", y, MLORA_F32, MLORA_STORE, xf, K, Wp, T, K, N)) return e;
  MLORA_CHECK(ks >= 1 && ks <= 4 && (ks == 1 || part) && (K / 32) / ks >= 1 && ((uintptr_t)xf & 15) == 0, MLORA_ERR_INVALID,
              "linear_ksplit_store: ks=%d outside 1..4, too many slices for K=%d, or no partials buffer", ks, K);
  if (T == 0) return MLORA_OK;
  if (T <= 64) return mlora_gemv_ksplit_store(y, part, ks, xf, Wp, T, K, N, stream);
  if (ks == 1) return mlora_linear_frag(y, MLORA_F32, MLORA_STORE, xf, Wp, T, K, N, stream);
  MidShape m = gemm_mid_shape(T, K, N, ks);
  m.ksplit = ks;                               // the caller's partial buffers were sized for ks slices
  const int e = launch_gemm_mid<OUT_F32>(y, part, N, m, (const elt*)xf, mlora_frag_tiles(T), (const elt*)Wp, T, K, N, (hipStream_t)stream);
  return e ? e : mlora_launch_status("linear_ksplit_store");
}
#endif

// K slices the mid-size kernel would use for resid [T, N] += xf . Wp^T with at most ks_max slices (T > 64)
int mlora_gemm_mid_ksplit(int T, int K, int N, int ks_max) { return gemm_mid_shape(T, K, N, ks_max).ksplit; }

// resid [T, N] fp32 += xf . Wp^T over ks K slices: slice 0 into resid, slices 1.. into part[ks - 1][T][ld_part] (T > 64)
int mlora_gemm_mid_acc(float* resid, float* part, int ld_part, int ks, const void* xf, const void* Wp, int T, int K, int N,
                       void* stream) {
  MLORA_CHECK(K % 32 == 0 && ks >= 1 && (K / 32) / ks >= 1 && ((uintptr_t)xf & 15) == 0, MLORA_ERR_UNSUPPORTED,
              "linear_frag (K slices): need K %% 32 == 0 and at least one 32-k step per slice (K=%d ks=%d)", K, ks);
  MidShape m = gemm_mid_shape(T, K, N, ks);
  m.ksplit = ks;                               // the caller's partial buffers were sized for ks slices
  const int e = launch_gemm_mid<OUT_ACC_F32>(resid, part, ld_part, m, (const elt*)xf, mlora_frag_tiles(T), (const elt*)Wp, T, K, N,
                                             (hipStream_t)stream);
  return e ? e : mlora_launch_status("linear_frag (K slices)");
}
