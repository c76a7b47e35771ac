// A prompt pass of the whole model enqueued natively: the operators of the per-operator path (llama.py, forward) in their order, with the same
// choices, from one call.  Up to a few hundred tokens a pass is shorter than the host takes to queue it operator by operator (14 us a launch; a
// launch from here 4): two layers of hidden 1024, 8 prompts of 27 to 54 tokens 422 -> 272 us, two of the 7B shape, 6 to 12 tokens 476 -> 365.
#include <initializer_list>

#include "common.h"

int mlora_check_attn(const char* who, int Hq, int Hkv, int D, int n_pages, int n_seq, int max_blocks);

namespace {

#define STEP(call)                   \
  do {                               \
    if (int e_ = (call)) return e_;  \
  } while (0)

// dst [n_rows, H] = rows of resid [T, H], to which the K-slice partials part[ks - 1][T][H] of the last linear are added first, in slice
// order (every row of resid is left with them).  A workgroup per row of resid; ks == 1: per row of dst, resid is only read.
__global__ __launch_bounds__(256) void take_rows_kernel(float* __restrict__ dst, float* __restrict__ resid, const float* __restrict__ part, int ks,
                                                        const long long* __restrict__ rows, int n_rows, int T, int H) {
  if (ks == 1) {
    const long long t = rows[blockIdx.x];
    if (t < 0 || t >= T) return;
    for (int c = threadIdx.x * 4; c < H; c += 1024)
      *reinterpret_cast<f32x4*>(dst + (size_t)blockIdx.x * H + c) = *reinterpret_cast<const f32x4*>(resid + (size_t)t * H + c);
    return;
  }
  const int t = blockIdx.x;
  for (int c = threadIdx.x * 4; c < H; c += 1024) {
    f32x4 v = *reinterpret_cast<const f32x4*>(resid + (size_t)t * H + c);
    for (int s = 0; s < ks - 1; ++s) v += *reinterpret_cast<const f32x4*>(part + ((size_t)s * T + t) * H + c);
    *reinterpret_cast<f32x4*>(resid + (size_t)t * H + c) = v;
    for (int i = 0; i < n_rows; ++i)
      if (rows[i] == t) *reinterpret_cast<f32x4*>(dst + (size_t)i * H + c) = v;
  }
}

size_t up256(size_t n) { return (n + 255) & ~(size_t)255; }

// How gate, up and their product are made in a layer
enum GateUp { GU_IL, GU_LINEAR, GU_STAGES, GU_DELTAS, GU_APART };       // out of the GEMV, the linear, the GEMM with LoRA stages, the linear with deltas; behind the linear
GateUp gate_up_form(const mlora_prefill_plan* p, const mlora_layer& L) {
  const int T = p->T, H = p->hidden, I = p->inter;
  const bool adapted = p->tok_adapter && (L.lora[MLORA_GATE].A || L.lora[MLORA_UP].A);
  if (T <= 64) return !adapted && L.gate_up_il_p ? GU_IL : GU_APART;
  if (!adapted) return GU_LINEAR;
  if (mlora_gemm_frag_preferred(T, H, 2 * I) && p->blk_adapter && !p->tok_rest) return GU_STAGES;
  return p->n_distinct > 0 && mlora_linear_frag_deltas_pay(T, H, 2 * I, 0, p->lora_r, p->n_distinct) ? GU_DELTAS : GU_APART;
}

// Where the intermediate results of a pass lie in its workspace (byte offsets).  q, k, v and the attention output are done with before gate and up are made, so
// their product (and they, where a layer keeps them) lies in the same place: 16384 tokens of the 7B shape 1.75 -> 0.67 GB, of which gate and up 0.72 that no layer wrote.
struct Slots {
  size_t xn, qkv, attn, gu, act, last, lora, lora_bytes, vsplit, ksplit, ksplit_bytes, total;
};
Slots slots_of(const mlora_prefill_plan* p) {
  const int T = p->T, H = p->hidden, I = p->inter, q_sz = p->n_q_heads * p->head_dim, qkv_sz = q_sz + 2 * p->n_kv_heads * p->head_dim;
  Slots s = {};
  size_t at = 0;
  auto take = [&](size_t bytes) { const size_t o = at; at += up256(bytes); return o; };
  s.xn = take(mlora_frag_activation_elems(T, H) * 2);
  const size_t shared = at;
  s.qkv = take((size_t)T * qkv_sz * 2);
  s.attn = take(mlora_frag_activation_elems(T, q_sz) * 2);
  const size_t attention_end = at;
  at = shared;
  s.act = take(mlora_frag_activation_elems(T, I) * 2);
  for (int l = 0; l < p->n_layers; ++l)
    if (gate_up_form(p, p->layers[l]) == GU_APART) {
      s.gu = take((size_t)T * 2 * I * 2);
      break;
    }
  at = at > attention_end ? at : attention_end;
  s.last = take((size_t)p->n_rows * H * 4 + mlora_frag_activation_elems(p->n_rows, H) * 2 + 256);
  if (p->tok_adapter) {
    for (int K : {H, q_sz, I}) {
      const size_t n = 3 * mlora_gather_mm_workspace_bytes(T, K, p->lora_r);
      s.lora_bytes = n > s.lora_bytes ? n : s.lora_bytes;
    }
    s.lora = take(s.lora_bytes);
    if (p->blk_adapter) s.vsplit = take((size_t)6 * up256((size_t)T * p->lora_r * 2));
  }
  if (T <= 256) {                                        // as the per-operator path: a short pass splits K of the two narrow linears
    s.ksplit_bytes = (size_t)3 * T * H * 4;
    s.ksplit = take(s.ksplit_bytes);
  }
  s.total = at;
  return s;
}

// A projection of a layer: its tables, and which rows of the (fused) weight it has
constexpr int MAXP = 3;
struct Proj {
  const mlora_lora_proj* t;
  int c0, n;
};
// the projections of in[0..n) that have tables
int live_of(const mlora_prefill_plan* p, const Proj* in, int n, Proj* out) {
  int live = 0;
  for (int i = 0; p->tok_adapter && i < n; ++i)
    if (in[i].t->A) out[live++] = in[i];
  return live;
}
// Whether the deltas of pj ride in the persistent GEMM as further k-steps: a 256-row block must lie in one projection
bool rides(const mlora_prefill_plan* p, int K, int N, const Proj* pj, int n) {
  bool r = n > 0 && p->blk_adapter && mlora_gemm_frag_preferred(p->T, K, N);
  for (int i = 0; i < n; ++i) r = r && pj[i].c0 % 256 == 0 && (pj[i].n % 256 == 0 || pj[i].c0 + pj[i].n == N);
  return r;
}

int check_plan(const mlora_prefill_plan* p) {
  MLORA_CHECK(p && p->layers, MLORA_ERR_INVALID, "prefill: null plan");
  MLORA_CHECK(p->T > 0 && p->n_layers >= 0 && p->n_rows > 0 && p->n_q_heads > 0 && p->n_kv_heads > 0 && p->head_dim > 0 && p->hidden > 0 && p->inter > 0 &&
                  p->vocab > 0,
              MLORA_ERR_INVALID, "prefill: bad sizes (T=%d rows=%d)", p->T, p->n_rows);
  MLORA_CHECK(p->hidden % 32 == 0 && p->inter % 32 == 0 && (p->n_q_heads * p->head_dim) % 32 == 0, MLORA_ERR_UNSUPPORTED,
              "prefill: hidden, intermediate and q sizes must be multiples of 32");
  MLORA_CHECK(!p->tok_adapter || p->lora_r == 8 || p->lora_r == 16 || p->lora_r == 32 || p->lora_r == 64, MLORA_ERR_UNSUPPORTED,
              "prefill: rank %d not in {8,16,32,64}", p->lora_r);
  MLORA_CHECK(!p->tok_adapter || (p->lora_n_ad > 0 && p->lora_n_ad <= 65535 && p->T <= (1 << 20)), MLORA_ERR_INVALID, "prefill: bad lora_n_ad %d (T=%d)",
              p->lora_n_ad, p->T);
  MLORA_CHECK(ceil_div(p->T, 128) <= 65535 && p->hidden <= 16384 && p->vocab % 4 == 0, MLORA_ERR_UNSUPPORTED,
              "prefill: T=%d or hidden=%d too large, or vocab %% 4 != 0 (%d)", p->T, p->hidden, p->vocab);
  MLORA_CHECK(!p->blk_adapter || (p->tok_adapter && (p->lora_r == 32 || p->lora_r == 64)), MLORA_ERR_INVALID, "prefill: blk_adapter goes with ranks 32 and 64");
  return MLORA_OK;
}

}  // namespace

extern "C" size_t mlora_prefill_workspace_bytes(const mlora_prefill_plan* p) { return check_plan(p) ? 0 : slots_of(p).total; }

extern "C" int mlora_prefill(const mlora_prefill_plan* p, void* stream) {
  STEP(check_plan(p));
  const int T = p->T, H = p->hidden, I = p->inter, Hq = p->n_q_heads, Hkv = p->n_kv_heads, D = p->head_dim;
  const int q_sz = Hq * D, kv_sz = Hkv * D, qkv_sz = q_sz + 2 * kv_sz;
  MLORA_CHECK(p->norm && p->lm_head_p && p->rope_cos && p->rope_sin && p->block_table && p->tok_seq && p->tok_pos && p->logits_rows && p->resid &&
                  p->logits && p->ws,
              MLORA_ERR_INVALID, "prefill: null buffer");
  const bool lora = p->tok_adapter != nullptr;
  // every layer, and what the operators ask of its sizes, is looked at before the first launch: a rejected call enqueues nothing
  STEP(mlora_check_attn("prefill", Hq, Hkv, D, p->n_pages, p->n_seq, p->max_blocks));
  MLORA_CHECK(T > 256 || H <= 8192 || (mlora_gemv_ksplit(T, q_sz, H) == 1 && mlora_gemv_ksplit(T, I, H) == 1), MLORA_ERR_UNSUPPORTED,
              "prefill: a pass that splits K needs hidden <= 8192 (%d)", H);
  for (int l = 0; l < p->n_layers; ++l) {
    const mlora_layer& L = p->layers[l];
    MLORA_CHECK(L.ln1 && L.ln2 && L.qkv_p && L.o_p && L.gate_up_p && L.down_p && L.k_cache && L.v_cache, MLORA_ERR_INVALID,
                "prefill: layer %d has a null weight, norm or cache pointer", l);
    for (int j = 0; lora && j < 7; ++j)
      MLORA_CHECK(!L.lora[j].A || L.lora[j].B, MLORA_ERR_INVALID, "prefill: layer %d projection %d has A but no B table", l, j);
    MLORA_CHECK(!lora || !p->segments || kv_sz % 16 == 0 || !(L.lora[MLORA_K].A || L.lora[MLORA_V].A), MLORA_ERR_UNSUPPORTED,
                "prefill: segments need key/value sizes in whole 16 (%d)", kv_sz);
    auto aligned = [&](int K, int N, std::initializer_list<Proj> all) {
      Proj pj[MAXP];
      const int n = live_of(p, all.begin(), (int)all.size(), pj);
      bool ok = true;
      for (int i = 0; rides(p, K, N, pj, n) && i < n; ++i) ok = ok && ((uintptr_t)pj[i].t->B & 15) == 0;
      return ok;
    };
    MLORA_CHECK(aligned(H, qkv_sz, {{&L.lora[MLORA_Q], 0, q_sz}, {&L.lora[MLORA_K], q_sz, kv_sz}, {&L.lora[MLORA_V], q_sz + kv_sz, kv_sz}}) &&
                    aligned(q_sz, H, {{&L.lora[MLORA_O], 0, H}}) && aligned(H, 2 * I, {{&L.lora[MLORA_GATE], 0, I}, {&L.lora[MLORA_UP], I, I}}) &&
                    aligned(I, H, {{&L.lora[MLORA_DOWN], 0, H}}),
                MLORA_ERR_INVALID, "prefill: layer %d: the B tables of deltas inside the persistent GEMM must be 16-byte aligned", l);
  }
  const Slots at = slots_of(p);
  MLORA_CHECK(p->ws_bytes >= at.total && ((uintptr_t)p->ws & 255) == 0, MLORA_ERR_WORKSPACE, "prefill: workspace of %zu bytes given, %zu needed (256-byte aligned)",
              p->ws_bytes, at.total);
  char* ws = (char*)p->ws;
  void *xn = ws + at.xn, *attn = ws + at.attn, *act = ws + at.act, *lora_ws = ws + at.lora;
  f16 *qkv = (f16*)(ws + at.qkv), *gu = (f16*)(ws + at.gu);
  float* part = at.ksplit_bytes ? (float*)(ws + at.ksplit) : nullptr;
  const int r = p->lora_r, n_ad = p->lora_n_ad;
  const float sc = p->lora_scaling;
  // deltas of projections that read x and own column ranges of y, for the tokens of ids
  struct Buckets { mlora_lora_bucket bk[MAXP]; int32_t c[MAXP], nc[MAXP]; };
  auto buckets_of = [&](const Proj* pj, int n) {
    Buckets b = {};
    for (int i = 0; i < n; ++i) {
      b.bk[i] = mlora_lora_bucket{pj[i].t->A, pj[i].t->B, r, n_ad, sc};
      b.c[i] = pj[i].c0;
      b.nc[i] = pj[i].n;
    }
    return b;
  };
  auto deltas = [&](void* y, int y_dtype, int ldy, const void* x, int K, const Proj* pj, int n, const int32_t* ids) -> int {
    if (n == 0) return MLORA_OK;
    const auto [bk, c, nc] = buckets_of(pj, n);
    if (p->segments)
      return mlora_gather_mm_segments(y, y_dtype, ldy, x, MLORA_FRAG, bk, n, c, nc, ids, T, K, lora_ws, at.lora_bytes, stream);
    if (n >= 2)
      return mlora_gather_mm_multi_proj(y, y_dtype, ldy, x, MLORA_FRAG, bk, 1, n, c, nc, nullptr, ids, T, K, lora_ws, at.lora_bytes, stream);
    return mlora_gather_mm((char*)y + (size_t)c[0] * (y_dtype == MLORA_F16 ? 2 : 4), y_dtype, ldy, x, MLORA_FRAG, bk[0].A, bk[0].B, ids, sc, T, K,
                           nc[0], r, n_ad, lora_ws, at.lora_bytes, stream);
  };
  // the shrink results of projections as fp16 halves, for a GEMM that carries their expand
  auto halves = [&](const void* x, int K, const Proj* pj, int n, mlora_fused_lora* out) -> int {
    void *hi[MAXP], *lo[MAXP];
    const void* A[MAXP];
    const size_t one = up256((size_t)T * r * 2);
    for (int i = 0; i < n; ++i) {
      hi[i] = ws + at.vsplit + (2 * i) * one;
      lo[i] = ws + at.vsplit + (2 * i + 1) * one;
      A[i] = pj[i].t->A;
      out[i] = mlora_fused_lora{pj[i].t->B, hi[i], lo[i], pj[i].c0, pj[i].n};
    }
    return mlora_lora_shrink_split(hi, lo, x, MLORA_FRAG, A, n, p->tok_adapter, sc, T, K, r, n_ad, lora_ws, at.lora_bytes, stream);
  };
  // y (=|+=) x . W^T with the deltas of pj: inside the GEMM where the shape has that form - of the persistent kernel for the blocks that agree
  // on an adapter, of the mid-size one for all where that pays.  ks (added
  // to fp32 only): the K slices whose partials the next norm adds.
  auto linear = [&](void* y, int y_dtype, int mode, const void* x, const void* W, int K, int N, const Proj* all, int n_all, int* ks) -> int {
    Proj pj[MAXP];
    const int n = live_of(p, all, n_all, pj);
    if (ks) *ks = 1;
    if (rides(p, K, N, pj, n)) {
      mlora_fused_lora f[MAXP];
      STEP(halves(x, K, pj, n, f));
      STEP(mlora_linear_frag_lora(y, y_dtype, mode, x, W, T, K, N, f, n, p->blk_adapter, r, stream));
      return p->tok_rest ? deltas(y, y_dtype, N, x, K, pj, n, p->tok_rest) : MLORA_OK;
    }
    if (n > 0 && p->n_distinct > 0 && (T > 64 || p->segments) && mlora_linear_frag_deltas_pay(T, K, N, mode == MLORA_ACCUMULATE, r, p->n_distinct)) {
      if (ks && part) {
        const int k = mlora_gemv_ksplit(T, K, N);
        *ks = k > 1 && mlora_gemv_ksplit_bytes(T, N, k) <= at.ksplit_bytes ? k : 1;
      }
      const Buckets b = buckets_of(pj, n);
      return mlora_linear_frag_deltas(y, y_dtype, mode, part, ks ? *ks : 1, x, W, T, K, N, b.bk, n, b.c, b.nc, p->tok_adapter, lora_ws, at.lora_bytes, stream);
    }
    if (ks && part) {
      const int riding = T <= 64 && n > 0 && !p->segments ? mlora_gemv_shrink_rows(K, 1, 1) : 0;
      const int k = mlora_gemv_ksplit(T, K, N + riding);
      *ks = k > 1 && mlora_gemv_ksplit_bytes(T, N, k) <= at.ksplit_bytes ? k : 1;
      STEP(mlora_gemv_frag_acc_ksplit((float*)y, nullptr, *ks > 1 ? part : nullptr, *ks, x, W, T, K, N, 0, nullptr, nullptr, 0, nullptr, 0, 0, stream));
    } else {
      STEP(mlora_linear_frag(y, y_dtype, mode, x, W, T, K, N, stream));
    }
    return deltas(y, y_dtype, N, x, K, pj, n, p->tok_adapter);
  };
  auto norm = [&](const void* w, int ks) -> int {
    if (ks > 1)
      return mlora_rmsnorm_ksplit(xn, MLORA_FRAG, p->resid, part, ks, H, w, p->eps, T, H, nullptr, 0, nullptr, nullptr, 0.f, 0, 0, 0, stream);
    return mlora_rmsnorm(xn, MLORA_FRAG, p->resid, MLORA_F32, w, p->eps, T, H, stream);
  };
  int ks = 1;
  for (int l = 0; l < p->n_layers; ++l) {
    const mlora_layer& L = p->layers[l];
    STEP(norm(L.ln1, ks));
    const Proj in[3] = {{&L.lora[MLORA_Q], 0, q_sz}, {&L.lora[MLORA_K], q_sz, kv_sz}, {&L.lora[MLORA_V], q_sz + kv_sz, kv_sz}};
    STEP(linear(qkv, MLORA_F16, MLORA_STORE, xn, L.qkv_p, H, qkv_sz, in, 3, nullptr));
    STEP(mlora_rope_kv_append(qkv, L.k_cache, L.v_cache, p->block_table, p->max_blocks, p->tok_seq, p->tok_pos, p->rope_cos, p->rope_sin, p->max_pos, T,
                              Hq, Hkv, D, p->n_pages, p->n_seq, stream));
    STEP(mlora_paged_attn_prefill(attn, MLORA_FRAG, qkv, L.k_cache, L.v_cache, p->block_table, p->max_blocks, p->tok_seq, p->tok_pos, T, Hq, Hkv, D,
                                  p->n_pages, p->n_seq, stream));
    const Proj o[1] = {{&L.lora[MLORA_O], 0, H}};
    STEP(linear(p->resid, MLORA_F32, MLORA_ACCUMULATE, attn, L.o_p, q_sz, H, o, 1, &ks));
    STEP(norm(L.ln2, ks));
    const Proj gate_up[2] = {{&L.lora[MLORA_GATE], 0, I}, {&L.lora[MLORA_UP], I, I}};
    Proj gl[MAXP];
    const int n_gl = live_of(p, gate_up, 2, gl);
    switch (gate_up_form(p, L)) {
      case GU_IL: STEP(mlora_gemv_frag_silu(act, xn, L.gate_up_il_p, T, H, I, stream)); break;
      case GU_LINEAR: STEP(mlora_linear_frag_glu(act, xn, L.gate_up_p, T, H, I, MLORA_GLU_SILU, 0.f, 0.f, 0.f, stream)); break;
      case GU_STAGES: {
        mlora_fused_lora f[MAXP];
        STEP(halves(xn, H, gl, n_gl, f));
        STEP(mlora_linear_frag_silu(act, xn, L.gate_up_p, T, H, I, f, n_gl, p->blk_adapter, r, stream));
        break;
      }
      case GU_DELTAS: {
        const Buckets b = buckets_of(gl, n_gl);
        STEP(mlora_linear_frag_silu_deltas(act, xn, L.gate_up_p, T, H, I, b.bk, n_gl, b.c, b.nc, p->tok_adapter, lora_ws, at.lora_bytes, stream));
        break;
      }
      case GU_APART:
        STEP(linear(gu, MLORA_F16, MLORA_STORE, xn, L.gate_up_p, H, 2 * I, gate_up, 2, nullptr));
        STEP(mlora_silu_mul(act, MLORA_FRAG, gu, gu + I, 2 * I, T, I, stream));
        break;
    }
    const Proj down[1] = {{&L.lora[MLORA_DOWN], 0, H}};
    STEP(linear(p->resid, MLORA_F32, MLORA_ACCUMULATE, act, L.down_p, I, H, down, 1, &ks));
  }
  float* last = (float*)(ws + at.last);
  void* last_n = ws + at.last + up256((size_t)p->n_rows * H * 4);
  hipLaunchKernelGGL(take_rows_kernel, dim3(ks > 1 ? T : p->n_rows), dim3(256), 0, (hipStream_t)stream, last, p->resid, part, ks, (const long long*)p->logits_rows,
                     p->n_rows, T, H);
  STEP(mlora_launch_status("prefill"));
  STEP(mlora_rmsnorm(last_n, MLORA_FRAG, last, MLORA_F32, p->norm, p->eps, p->n_rows, H, stream));
  return mlora_linear_frag(p->logits, MLORA_F32, MLORA_STORE, last_n, p->lm_head_p, p->n_rows, H, p->vocab, stream);
}
