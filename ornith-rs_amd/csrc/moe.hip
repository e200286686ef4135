// The sparse MoE block: router softmax + top-k, expert FFNs, shared expert, tail.
//
// Replaces moe::sparse_moe_block and its helpers
// (/root/reference/src/ops/moe.rs:113-134,256-338,548-596,662-741) and the
// kernels router_top_k / moe_combine / swiglu
// (/root/reference/kernels/moe.metal:207-258,568-614,
//  /root/reference/kernels/ornith_elementwise.metal:97-105) and the vendored
// precise softmax (softmax.h:10-98).
//
// Rounding points are the reference's: gates, probabilities, every expert output
// and every step of the tail are bf16; sums inside a kernel are fp32.
#include "linear_device.h"
#include "mm_narrow_host.h"
#include "moe_device.h"
#include "norm_device.h"
#include "rt.h"

// linear.hip
extern "C" int dense_gather_mv_multi(ornith_ctx* ctx, const void* const* d_ws, int n, int E, int O, int K,
                                     const void* d_x, int x_rows, const uint32_t* d_lhs,
                                     const uint32_t* d_rhs, int rows, void* const* d_ys);
int linear_exact_multi(ornith_ctx* ctx, const ornith_linear* const* ws, int n, const void* d_x, int M, void* const* d_ys);
// moe_fused.hip
bool moe_fused_supported(const ornith_moe_weights* w);
bool moe_fused_router(ornith_ctx* ctx, const ornith_moe_weights* w, const void* d_x, int T,
                      void* d_gates, void* d_egate, int* rc, const PreNorm* pre);
bool moe_one_launch(ornith_ctx* ctx, const ornith_moe_weights* w, const void* d_x, int T, void* d_gates,
                    void* d_egate, uint32_t* d_inds, void* d_scores, void* d_act, void* d_out,
                    const PreNorm* pre, int* rc);
// moe_affine4.hip: the expert half for routed and shared experts in 4-bit affine group 32
bool moe_affine4_supported(const ornith_moe_weights* w);
int moe_affine4_experts(ornith_ctx* ctx, const ornith_moe_weights* w, const void* d_x, int T, const uint32_t* d_inds,
                        const void* d_scores, const void* d_egate, void* d_act, void* d_out, const void* d_gates);
// ... and for dense bf16 experts (the MTP head's block)
bool moe_dense_supported(const ornith_moe_weights* w);
int moe_dense_experts(ornith_ctx* ctx, const ornith_moe_weights* w, const void* d_x, int T, const uint32_t* d_inds,
                      const void* d_scores, const void* d_egate, void* d_act, void* d_out, const void* d_gates);
// kq_mm.hip
size_t moe_plan_bytes(int pairs, int E, int rows, int shared_rows);
int moe_plan(ornith_ctx* ctx, const uint32_t* d_inds, int pairs, int E, int rows, int shared_rows, void* d_plan, bool build,
             nmm::Plan* out);
int moe_fused_experts(ornith_ctx* ctx, const ornith_moe_weights* w, const void* d_x, int T,
                      const uint32_t* d_inds, const void* d_scores, const void* d_egate, void* d_act,
                      void* d_out, int phases, const void* d_gates);

namespace {

// One wavefront per token. Lane l holds gates [l*PER, (l+1)*PER).
//   softmax: fp32 max, e = exp(g - max), lane-sequential sum then butterfly,
//            p = bf16(e * (1/sum))
//   top-k:   k rounds of (value, then larger index) selection; round r -> slot k-1-r
// Also writes the gather index lists the expert mat-vecs use:
//   lhs_tok[t*k+j] = t (row of x), lhs_row[t*k+j] = t*k+j (row of act).
template <int PER>
__global__ __launch_bounds__(64) void router_topk_kernel(const bf16_t* gates, int E, int k,
                                                         uint32_t* inds, bf16_t* scores,
                                                         bf16_t* probs, uint32_t* lhs_tok,
                                                         uint32_t* lhs_row) {
  const int t = blockIdx.x, lane = threadIdx.x;
  router_topk_wave<PER>(gates + (size_t)t * E, k, inds + (size_t)t * k, scores + (size_t)t * k,
                        probs ? probs + (size_t)t * E : nullptr, lane);
  if (lane < k) {
    if (lhs_tok) lhs_tok[t * k + lane] = t;
    if (lhs_row) lhs_row[t * k + lane] = t * k + lane;
  }
}

// The router's tail at prefill widths, one wavefront a token: the shared expert's gate (one affine
// row dot, its loads ahead of the softmax's arithmetic) and softmax + top-k.
struct EgateArgs {
  const uint8_t* w;
  const bf16_t *s, *b, *x;
  bf16_t* y;
  int K, bits;  // bits 0: not made here
};
template <int PER>
__global__ __launch_bounds__(64) void router_egate_kernel(const bf16_t* gates, int E, int k, uint32_t* inds,
                                                          bf16_t* scores, EgateArgs g) {
  const int t = blockIdx.x, lane = threadIdx.x;
  if (g.bits) {
    const bf16_t* xr = g.x + (size_t)t * g.K;
    const float v = g.bits == 8 ? affine8_row_dot(g.w, g.s, g.b, xr, g.K, lane) : affine4_row_dot(g.w, g.s, g.b, xr, g.K, lane);
    if (lane == 0) g.y[t] = dm_f2bf(v);
  }
  router_topk_wave<PER>(gates + (size_t)t * E, k, inds + (size_t)t * k, scores + (size_t)t * k, nullptr, lane);
}

// V consecutive elements a thread (V = 8: 16-byte loads and stores; V = 1 for odd sizes)
template <int V>
struct BfPack;
template <>
struct BfPack<8> { typedef unsigned int type __attribute__((ext_vector_type(4))); };
template <>
struct BfPack<1> { typedef bf16_t type; };
template <int V>
__device__ __forceinline__ float bf_get(const typename BfPack<V>::type& p, int i) {
  if constexpr (V == 1) return dm_bf2f(p);
  else return (i & 1) ? dm_bf2f_hi(p[i >> 1]) : dm_bf2f_lo(p[i >> 1]);
}
template <int V>
__device__ __forceinline__ void bf_put(typename BfPack<V>::type& p, int i, float v) {
  if constexpr (V == 1) p = dm_f2bf(v);
  else p[i >> 1] = (i & 1) ? (p[i >> 1] & 0xffffu) | ((uint32_t)dm_f2bf(v) << 16) : (uint32_t)dm_f2bf(v);
}

template <int V>
__global__ void swiglu_kernel(const bf16_t* gate, const bf16_t* up, bf16_t* out, int64_t n,
                              const bf16_t* gate2 = nullptr, const bf16_t* up2 = nullptr,
                              bf16_t* out2 = nullptr, int64_t n2 = 0) {
  typedef typename BfPack<V>::type P;
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  // a second, independent range follows the first (two activations in one launch)
  if (i >= n / V) {
    i -= n / V;
    if (i >= n2 / V) return;
    gate = gate2;
    up = up2;
    out = out2;
  }
  const P g8 = reinterpret_cast<const P*>(gate)[i], u8 = reinterpret_cast<const P*>(up)[i];
  P o8;
#pragma unroll
  for (int e = 0; e < V; ++e) {
    const float g = bf_get<V>(g8, e);
    const float s = dm_rb(g * dm_sigmoid_bf16(g));
    bf_put<V>(o8, e, s * bf_get<V>(u8, e));
  }
  reinterpret_cast<P*>(out)[i] = o8;
}

// V output elements (from c on) of token t: j ascends, every step rounds to bf16. Bound by the stream at long prompts, by one trip
// to memory at short ones: eight experts' rows, their scores and the rest are asked for at once (past k the last one again,
// unused), and nothing is divided but by the workgroup. With the scores added up one load after the other ahead of the rows, us, 51 / 700 /
// 6621 tokens: 5.3 / 10.3 / 62.4 -> 5.0 / 8.3 / 53. `more` asks for what the caller needs besides.
struct CombineArgs {
  const bf16_t *scores, *y, *gate, *shared;
  int T, k, dim, normalize;
};
template <int V, class F>
__device__ __forceinline__ typename BfPack<V>::type combine_row(const CombineArgs& a, uint32_t t, uint32_t c, F more) {
  typedef typename BfPack<V>::type P;
  const int k = a.k;
  const bf16_t* s = a.scores + (size_t)t * k;
  P yj[8];
  bf16_t sj[8];
  auto fetch = [&](int j0) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      yj[j] = *reinterpret_cast<const P*>(a.y + ((size_t)t * k + min(j0 + j, k - 1)) * a.dim + c);
      sj[j] = s[min(j0 + j, k - 1)];
    }
  };
  fetch(0);
  const P sh = *reinterpret_cast<const P*>(a.shared + (size_t)t * a.dim + c);
  const bf16_t gt = a.gate[t];
  more();
  float denom = 0.f;
  if (a.normalize) {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (j < k) denom = dm_rb(dm_bf2f(sj[j]) + denom);
    for (int j = 8; j < k; ++j) denom = dm_rb(dm_bf2f(s[j]) + denom);
  }
  float acc[V];
#pragma unroll
  for (int e = 0; e < V; ++e) acc[e] = 0.f;
  for (int j0 = 0;;) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (j0 + j >= k) break;
      const float w = a.normalize ? dm_rb(dm_bf2f(sj[j]) / denom) : dm_bf2f(sj[j]);
#pragma unroll
      for (int e = 0; e < V; ++e) {
        const float weighted = dm_rb(bf_get<V>(yj[j], e) * w);
        acc[e] = dm_rb(weighted + acc[e]);
      }
    }
    j0 += 8;
    if (j0 >= k) break;
    fetch(j0);
  }
  const float g = dm_sigmoid_bf16(dm_bf2f(gt));
  P o;
#pragma unroll
  for (int e = 0; e < V; ++e) {
    const float gated = dm_rb(g * bf_get<V>(sh, e));
    bf_put<V>(o, e, acc[e] + gated);
  }
  return o;
}
// (arguments one by one: a struct's come by a scalar load, 0.3 us of 4.5 at 300 rows of 2048 values)
template <int V>
__global__ __launch_bounds__(256) void moe_combine_kernel(const bf16_t* scores, const bf16_t* y, const bf16_t* gate, const bf16_t* shared,
                                                          bf16_t* out, int T, int k, int dim, int normalize) {
  const CombineArgs a{scores, y, gate, shared, T, k, dim, normalize};
  // (a grid has fewer than 2^32 threads)
  const uint32_t per_row = a.dim / V, base = blockIdx.x * 256u, t0 = base / per_row;
  uint32_t r = base - t0 * per_row + threadIdx.x, t = t0;
  if (per_row >= 256u) {
    if (r >= per_row) {
      r -= per_row;
      ++t;
    }
  } else {
    t += r / per_row;
    r %= per_row;
  }
  if (t >= (uint32_t)a.T) return;
  *reinterpret_cast<typename BfPack<V>::type*>(out + (size_t)t * a.dim + r * V) = combine_row<V>(a, t, r * V, []() {});
}
// The same with what follows a block in the model, h = res + out and rms_norm(h): a workgroup of 8 * PER threads a token of 64 * PER values,
// eight a thread, and the block's output goes nowhere. Bound as the combine is: the norm's streams hide in its wait. The two launches
// and this one, us, 700 / 6621 tokens of 2048 values: 8.3 + 5.0 / 56 + 18.5 -> 10.4 / 65.7 (a layer; a prompt of 51: 6.37 -> 6.25 ms).
template <int PER>
__global__ __launch_bounds__(PER * 8) void moe_combine_norm_kernel(CombineArgs a, PreNorm n) {
  __shared__ float sums[64];
  const uint32_t t = blockIdx.x, c = 8 * threadIdx.x;
  const size_t at = (size_t)t * a.dim + c;
  float x[8], w[8];
  const auto o = combine_row<8>(a, t, c, [&]() {
    load_bf16<8>(n.res + at, x);
    load_bf16<8>(n.w + c, w);
  });
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i] = dm_rb(x[i] + bf_get<8>(o, i));
  store_bf16<8>(n.h_out + at, x);
  const float inv = wide_row_inv<PER>(x, a.dim, n.eps, sums);
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i] = dm_rb(w[i] * dm_rb(x[i] * inv));
  store_bf16<8>(n.normed_out + at, x);
}

int launch_router(ornith_ctx* ctx, const bf16_t* gates, int T, int E, int k, uint32_t* inds,
                  bf16_t* scores, bf16_t* probs, uint32_t* lhs_tok, uint32_t* lhs_row) {
#define ROUTER_CASE(P)                                                                       \
  case P:                                                                                    \
    hipLaunchKernelGGL(router_topk_kernel<P>, dim3(T), dim3(64), 0, ctx->stream, gates, E, k, \
                       inds, scores, probs, lhs_tok, lhs_row);                               \
    break;
  switch (E % 64 == 0 ? E / 64 : 0) {
    ROUTER_CASE(1)
    ROUTER_CASE(2)
    ROUTER_CASE(4)
    ROUTER_CASE(8)
    ROUTER_CASE(16)
    default:
      return ornith_fail(ORNITH_ERR_UNSUPPORTED, "router_topk: E=%d (need 64,128,256,512,1024)", E);
  }
#undef ROUTER_CASE
  ORN_LAUNCH_CHECK("router_topk_kernel");
  return ORNITH_OK;
}

int launch_router_egate(ornith_ctx* ctx, const bf16_t* gates, int T, int E, int k, uint32_t* inds, bf16_t* scores,
                        const ornith_linear& w, const bf16_t* x, bf16_t* egate) {
  EgateArgs g{};
  if (w.mode == ORNITH_LIN_AFFINE8 || w.mode == ORNITH_LIN_AFFINE4) {
    ORN_REQUIRE(w.d_w && w.d_scales && w.d_biases && w.K % 64 == 0, "moe_block: shared expert gate K=%d", w.K);
    g = {(const uint8_t*)w.d_w, (const bf16_t*)w.d_scales, (const bf16_t*)w.d_biases, x, egate, w.K, w.mode == ORNITH_LIN_AFFINE8 ? 8 : 4};
  } else {
    const int rc = ornith_linear_matmul(ctx, &w, x, T, egate);
    if (rc) return rc;
  }
#define ROUTER_CASE(P)                                                                                         \
  case P:                                                                                                      \
    hipLaunchKernelGGL(router_egate_kernel<P>, dim3(T), dim3(64), 0, ctx->stream, gates, E, k, inds, scores, g); \
    break;
  switch (E % 64 == 0 ? E / 64 : 0) {
    ROUTER_CASE(1)
    ROUTER_CASE(2)
    ROUTER_CASE(4)
    ROUTER_CASE(8)
    ROUTER_CASE(16)
    default:
      return ornith_fail(ORNITH_ERR_UNSUPPORTED, "router_topk: E=%d (need 64,128,256,512,1024)", E);
  }
#undef ROUTER_CASE
  ORN_LAUNCH_CHECK("router_egate_kernel");
  return ORNITH_OK;
}

// The block's last launch: the combine, with `close` the sum and norm that follow it too where the shapes allow (*close->done says so; d_out is
// not written then).
int combine_and_close(ornith_ctx* ctx, const void* scores, const void* y, const void* gate, const void* shared, int T, int k, int dim,
                      int normalize, void* d_out, MoeClose* close) {
  if (close && (dim == 1024 || dim == 2048 || dim == 4096)) {
    const PreNorm& n = close->norm;
    const uintptr_t all = (uintptr_t)y | (uintptr_t)shared | (uintptr_t)n.res | (uintptr_t)n.w | (uintptr_t)n.h_out | (uintptr_t)n.normed_out;
    if ((all & 15) == 0) {
      const CombineArgs a{(const bf16_t*)scores, (const bf16_t*)y, (const bf16_t*)gate, (const bf16_t*)shared, T, k, dim, normalize};
      if (dim == 1024) hipLaunchKernelGGL(moe_combine_norm_kernel<16>, dim3(T), dim3(128), 0, ctx->stream, a, n);
      else if (dim == 2048) hipLaunchKernelGGL(moe_combine_norm_kernel<32>, dim3(T), dim3(256), 0, ctx->stream, a, n);
      else hipLaunchKernelGGL(moe_combine_norm_kernel<64>, dim3(T), dim3(512), 0, ctx->stream, a, n);
      ORN_LAUNCH_CHECK("moe_combine_norm_kernel");
      close->done = true;
      return ORNITH_OK;
    }
  }
  return ornith_moe_combine(ctx, scores, y, gate, shared, T, k, dim, normalize, d_out);
}

// Prompts of few rows an expert (and a layer's prompt over affine experts, which have no wide form): the
// shared expert is one more expert of the pair list, so the block is six launches: router, its
// tail (shared gate, softmax + top-k), plan, gate + up + swiglu, down, combine.
// false: the shapes are not covered.
bool moe_block_narrow(ornith_ctx* ctx, const ornith_moe_weights* w, const void* d_x, int T, void* d_out, MoeClose* close, int* rc_out) {
  const int E = w->router.O, H = w->router.K, I = w->ex_gate.O, k = w->top_k, pairs = T * k;
  if (E % 64 != 0 || E > 1024) return false;
  const int rows = nmm::tile_rows(pairs, E);
  const size_t plan_bytes = moe_plan_bytes(pairs, E, rows, T);
  const size_t need = 2 * ((size_t)T * E + T + (size_t)(pairs + T) * (I + H) + (size_t)pairs) + 4 * (size_t)pairs + plan_bytes + 16 * 256;
  void* base = nullptr;
  int rc = *rc_out = ornith_scratch(ctx, need, &base);
  if (rc) return true;
  ScratchCursor sc(base);
  bf16_t* gates = sc.take<bf16_t>((size_t)T * E);
  uint32_t* inds = sc.take<uint32_t>(pairs);
  bf16_t* scores = sc.take<bf16_t>(pairs);
  bf16_t* eg = sc.take<bf16_t>(T);
  bf16_t* act = sc.take<bf16_t>((size_t)(pairs + T) * I);
  bf16_t* y = sc.take<bf16_t>((size_t)(pairs + T) * H);
  void* plan = sc.take<char>(plan_bytes);
  if (!nmm::moe_ok(w, d_x, T, act, y)) return false;
  nmm::Plan pl;
  auto go = [&]() -> int {
#define TRY(e)          \
  do {                  \
    rc = (e);           \
    if (rc) return rc;  \
  } while (0)
    TRY(ornith_linear_matmul(ctx, &w->router, d_x, T, gates));
    TRY(launch_router_egate(ctx, gates, T, E, k, inds, scores, w->sh_egate, (const bf16_t*)d_x, eg));
    TRY(moe_plan(ctx, inds, pairs, E, rows, T, plan, true, &pl));
    TRY(nmm::gate_up(ctx, w, d_x, pairs, pl, act));
    TRY(nmm::gathered(ctx, &w->ex_down, &w->sh_down, act, pairs, 1, pl, y));
    TRY(combine_and_close(ctx, scores, y, eg, y + (size_t)pairs * H, T, k, H, w->norm_topk_prob, d_out, close));
#undef TRY
    return ORNITH_OK;
  };
  *rc_out = go();
  return true;
}

// Prefill widths: the same block with every projection as a matrix-core GEMM and the routed
// experts as three expert-grouped GEMMs over one sorted pair list
// (/root/reference/src/ops/moe.rs:662-741 at T above the exact window; gather_qmm_t).
int moe_block_prefill(ornith_ctx* ctx, const ornith_moe_weights* w, const void* d_x, int T, void* d_out, MoeClose* close) {
  const int E = w->router.O, H = w->router.K, I = w->ex_gate.O, k = w->top_k, SI = w->sh_gate.O;
  const int pairs = T * k;
  const size_t plan_bytes = ornith_kq_gather_plan_bytes(pairs, E);
  const size_t need = 2 * ((size_t)T * E + (size_t)T * SI * 3 + (size_t)T * H + T + (size_t)pairs * (3 * I + H) +
                           (size_t)pairs) + 4 * (size_t)pairs + plan_bytes + 24 * 256;
  void* base = nullptr;
  int rc = ornith_scratch(ctx, need, &base);
  if (rc) return rc;
  ScratchCursor sc(base);
  bf16_t* gates = sc.take<bf16_t>((size_t)T * E);
  uint32_t* inds = sc.take<uint32_t>(pairs);
  bf16_t* scores = sc.take<bf16_t>(pairs);
  bf16_t* sg = sc.take<bf16_t>((size_t)T * SI);
  bf16_t* su = sc.take<bf16_t>((size_t)T * SI);
  bf16_t* sact = sc.take<bf16_t>((size_t)T * SI);
  bf16_t* sy = sc.take<bf16_t>((size_t)T * H);
  bf16_t* eg = sc.take<bf16_t>(T);
  bf16_t* xg = sc.take<bf16_t>((size_t)pairs * I);
  bf16_t* xu = sc.take<bf16_t>((size_t)pairs * I);
  bf16_t* act = sc.take<bf16_t>((size_t)pairs * I);
  bf16_t* y = sc.take<bf16_t>((size_t)pairs * H);
  void* plan = sc.take<char>(plan_bytes);
#define TRY(e)          \
  do {                  \
    rc = (e);           \
    if (rc) return rc;  \
  } while (0)
  {
    // the router and the shared expert's gate / up read the same rows: one launch where their
    // formats allow (alone, the 256-column router is 64 workgroups)
    const ornith_linear* in3[3] = {&w->router, &w->sh_gate, &w->sh_up};
    void* y3[3] = {gates, sg, su};
    TRY(ornith_linear_matmul_multi(ctx, in3, 3, d_x, T, y3));
  }
  TRY(ornith_linear_matmul(ctx, &w->sh_egate, d_x, T, eg));
  TRY(launch_router(ctx, gates, T, E, k, inds, scores, nullptr, nullptr, nullptr));
  TRY(ornith_swiglu(ctx, sg, su, (int64_t)T * SI, sact));
  TRY(ornith_linear_matmul(ctx, &w->sh_down, sact, T, sy));
  TRY(ornith_kq_gather_matmul(ctx, &w->ex_gate, d_x, inds, pairs, k, 1, plan, 1, xg));
  TRY(ornith_kq_gather_matmul(ctx, &w->ex_up, d_x, inds, pairs, k, 1, plan, 0, xu));
  TRY(ornith_swiglu(ctx, xg, xu, (int64_t)pairs * I, act));
  TRY(ornith_kq_gather_matmul(ctx, &w->ex_down, act, inds, pairs, k, 0, plan, 0, y));
  TRY(combine_and_close(ctx, scores, y, eg, sy, T, k, H, w->norm_topk_prob, d_out, close));
#undef TRY
  return ORNITH_OK;
}

}  // namespace

extern "C" {

int ornith_router_topk(ornith_ctx* ctx, const void* d_gates, int T, int E, int k, uint32_t* d_inds,
                       void* d_scores, void* d_probs) {
  ORN_REQUIRE(ctx && d_gates && d_inds && d_scores, "router_topk: null argument");
  ORN_REQUIRE(T >= 1 && E % 64 == 0 && k >= 1 && k <= 16 && k <= E, "router_topk: T=%d E=%d k=%d",
              T, E, k);
  return launch_router(ctx, (const bf16_t*)d_gates, T, E, k, d_inds, (bf16_t*)d_scores,
                       (bf16_t*)d_probs, nullptr, nullptr);
}

int ornith_swiglu(ornith_ctx* ctx, const void* d_gate, const void* d_up, int64_t n, void* d_out) {
  ORN_REQUIRE(ctx && d_gate && d_up && d_out && n >= 0, "swiglu: bad argument");
  if (n == 0) return ORNITH_OK;
  // 16-byte pieces when the size and the addresses allow
  if (n % 8 == 0 && (((uintptr_t)d_gate | (uintptr_t)d_up | (uintptr_t)d_out) & 15) == 0)
    hipLaunchKernelGGL(swiglu_kernel<8>, dim3((unsigned)((n / 8 + 255) / 256)), dim3(256), 0, ctx->stream,
                       (const bf16_t*)d_gate, (const bf16_t*)d_up, (bf16_t*)d_out, n);
  else
    hipLaunchKernelGGL(swiglu_kernel<1>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, ctx->stream,
                       (const bf16_t*)d_gate, (const bf16_t*)d_up, (bf16_t*)d_out, n);
  ORN_LAUNCH_CHECK("swiglu_kernel");
  return ORNITH_OK;
}

}  // extern "C"

// swiglu over two independent ranges in one launch
static int swiglu_pair(ornith_ctx* ctx, const void* g1, const void* u1, int64_t n1, void* o1, const void* g2,
                       const void* u2, int64_t n2, void* o2) {
  ORN_REQUIRE(g1 && u1 && o1 && g2 && u2 && o2 && n1 >= 0 && n2 >= 0, "swiglu_pair: bad argument");
  if (n1 + n2 == 0) return ORNITH_OK;
  const uintptr_t bits = (uintptr_t)g1 | (uintptr_t)u1 | (uintptr_t)o1 | (uintptr_t)g2 | (uintptr_t)u2 | (uintptr_t)o2;
  if (n1 % 8 == 0 && n2 % 8 == 0 && (bits & 15) == 0)
    hipLaunchKernelGGL(swiglu_kernel<8>, dim3((unsigned)(((n1 + n2) / 8 + 255) / 256)), dim3(256), 0, ctx->stream,
                       (const bf16_t*)g1, (const bf16_t*)u1, (bf16_t*)o1, n1, (const bf16_t*)g2,
                       (const bf16_t*)u2, (bf16_t*)o2, n2);
  else
    hipLaunchKernelGGL(swiglu_kernel<1>, dim3((unsigned)((n1 + n2 + 255) / 256)), dim3(256), 0, ctx->stream,
                       (const bf16_t*)g1, (const bf16_t*)u1, (bf16_t*)o1, n1, (const bf16_t*)g2,
                       (const bf16_t*)u2, (bf16_t*)o2, n2);
  ORN_LAUNCH_CHECK("swiglu_kernel<pair>");
  return ORNITH_OK;
}

extern "C" {

int ornith_moe_combine(ornith_ctx* ctx, const void* d_scores, const void* d_y, const void* d_gate,
                       const void* d_shared, int T, int k, int dim, int normalize, void* d_out) {
  ORN_REQUIRE(ctx && d_scores && d_y && d_gate && d_shared && d_out, "moe_combine: null argument");
  ORN_REQUIRE(T >= 1 && k >= 1 && dim >= 1, "moe_combine: T=%d k=%d dim=%d", T, k, dim);
  const int64_t n = (int64_t)T * dim;
  const bool wide = dim % 8 == 0 && (((uintptr_t)d_y | (uintptr_t)d_shared | (uintptr_t)d_out) & 15) == 0;
  const int64_t threads = wide ? n / 8 : n;
  hipLaunchKernelGGL(wide ? moe_combine_kernel<8> : moe_combine_kernel<1>, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, ctx->stream,
                     (const bf16_t*)d_scores, (const bf16_t*)d_y, (const bf16_t*)d_gate, (const bf16_t*)d_shared, (bf16_t*)d_out, T, k, dim, normalize);
  ORN_LAUNCH_CHECK("moe_combine_kernel");
  return ORNITH_OK;
}

// The block. With `pre`, x is rms_norm(pre->res + pre->y): made inside the router launch when
// the fused kernels cover the shapes (d_x then is where the normed rows get stored, and read
// back by the expert kernels), by a separate add_rms_norm otherwise.
// `gemm_affine`: a prompt's rows may run as GEMMs over affine experts too. It belongs to the entry
// point, not to the outputs asked for: ornith_moe_block, which gives ids and scores on demand, keeps
// these experts exact at every width, so that asking does not change the result.
static int moe_block_impl(ornith_ctx* ctx, const ornith_moe_weights* w, const void* d_x, int T,
                          void* d_out, uint32_t* d_inds_out, void* d_scores_out, const PreNorm* pre, bool gemm_affine,
                          MoeClose* close = nullptr) {
  ORN_REQUIRE(ctx && w && d_x && d_out, "moe_block: null argument");
  const int E = w->router.O, H = w->router.K, I = w->ex_gate.O, k = w->top_k;
  ORN_REQUIRE(T >= 1 && T <= 8192, "moe_block: T=%d", T);
  ORN_REQUIRE(k >= 1 && k <= 16 && k <= E, "moe_block: top_k=%d of %d", k, E);
  ORN_REQUIRE(w->ex_gate.E == E && w->ex_up.E == E && w->ex_down.E == E,
              "moe_block: expert tensors carry %d/%d/%d experts, router has %d", w->ex_gate.E,
              w->ex_up.E, w->ex_down.E, E);
  ORN_REQUIRE(w->ex_gate.K == H && w->ex_up.K == H && w->ex_up.O == I && w->ex_down.K == I &&
                  w->ex_down.O == H,
              "moe_block: expert shapes do not chain (H=%d I=%d)", H, I);
  ORN_REQUIRE(w->sh_gate.K == H && w->sh_up.K == H && w->sh_up.O == w->sh_gate.O &&
                  w->sh_down.K == w->sh_gate.O && w->sh_down.O == H && w->sh_egate.K == H &&
                  w->sh_egate.O == 1,
              "moe_block: shared expert shapes do not chain");
  const int SI = w->sh_gate.O;
  const bool pre_in_kernel = pre && T <= 4 && T < kPrefillRows && H == kPreN && prenorm_apart(*pre, T) && ornith_option_fuse_norm() &&
                             ornith_option_fuse_moe() && moe_fused_supported(w) &&
                             w->router.mode == ORNITH_LIN_KQUANT;
  // (an affine block's router and shared-expert gate take it in the head of their launch, below)
  const bool ex_affine4 = !w->ex_dense && w->ex_gate.kind == ORNITH_AFFINE4_G32;
  const bool pair_a4 = ex_affine4 && moe_affine4_supported(w);
  const bool pre_in_a4 = pre && T <= 4 && T < kPrefillRows && ornith_option_fuse_moe() && pair_a4;
  if (pre && !pre_in_kernel && !pre_in_a4) {
    int rcn = ornith_add_rms_norm(ctx, pre->res, pre->y, pre->w, T, H, pre->eps, pre->h_out, pre->normed_out);
    if (rcn) return rcn;
    pre = nullptr;
  }
  if (ex_affine4)
    ORN_REQUIRE(w->ex_up.kind == ORNITH_AFFINE4_G32 && w->ex_down.kind == ORNITH_AFFINE4_G32,
                "moe_block: the three expert stacks must share the 4-bit affine format");
  if (T >= kPrefillRows && !w->ex_dense && (ex_affine4 ? gemm_affine : !d_inds_out && !d_scores_out)) {
    int rcn = ORNITH_OK;
    if (moe_block_narrow(ctx, w, d_x, T, d_out, close, &rcn)) return rcn;
  }
  if (T >= kPrefillRows && !w->ex_dense && !ex_affine4) {
    ORN_REQUIRE(!d_inds_out && !d_scores_out, "moe_block: index outputs are a decode-width feature");
    return moe_block_prefill(ctx, w, d_x, T, d_out, close);
  }
  // dense experts have no prefill-width form, affine ones none that is exact: the rows go in blocks
  // of 64 (they are independent of each other, so the result is the same)
  if (T > 64) {
    for (int t0 = 0; t0 < T; t0 += 64) {
      const int n = T - t0 < 64 ? T - t0 : 64;
      const int rcb = moe_block_impl(ctx, w, static_cast<const bf16_t*>(d_x) + (size_t)t0 * H, n,
                                     static_cast<bf16_t*>(d_out) + (size_t)t0 * H,
                                     d_inds_out ? d_inds_out + (size_t)t0 * k : nullptr,
                                     d_scores_out ? static_cast<bf16_t*>(d_scores_out) + (size_t)t0 * k : nullptr, nullptr, false);
      if (rcb) return rcb;
    }
    return ORNITH_OK;
  }

  const size_t need = 2 * ((size_t)T * E * 2 + (size_t)T * SI * 3 + (size_t)T * H + T +
                           (size_t)(T * k + T) * (2 * I + I + SI + H + 1)) +
                      4 * (size_t)T * k * 3 + 64 * 256;
  void* base = nullptr;
  int rc = ornith_scratch(ctx, need, &base);
  if (rc) return rc;
  ScratchCursor sc(base);
  bf16_t* gates = sc.take<bf16_t>((size_t)T * E);
  // the routing goes straight where the caller wants it (copies behind the block were 2.7 us of 19.6)
  uint32_t* inds = d_inds_out ? d_inds_out : sc.take<uint32_t>((size_t)T * k);
  bf16_t* scores = d_scores_out ? static_cast<bf16_t*>(d_scores_out) : sc.take<bf16_t>((size_t)T * k);
  uint32_t* lhs_tok = sc.take<uint32_t>((size_t)T * k);
  uint32_t* lhs_row = sc.take<uint32_t>((size_t)T * k);
  bf16_t* sg = sc.take<bf16_t>((size_t)T * SI);
  bf16_t* su = sc.take<bf16_t>((size_t)T * SI);
  bf16_t* sact = sc.take<bf16_t>((size_t)T * SI);
  bf16_t* sy = sc.take<bf16_t>((size_t)T * H);
  bf16_t* eg = sc.take<bf16_t>((size_t)T);
  bf16_t* xg = sc.take<bf16_t>((size_t)T * k * I);
  bf16_t* xu = sc.take<bf16_t>((size_t)T * k * I);
  bf16_t* act = sc.take<bf16_t>((size_t)(T * k + T) * (I > SI ? I : SI));
  bf16_t* y = sc.take<bf16_t>((size_t)T * k * H);

#define TRY(e)          \
  do {                  \
    rc = (e);           \
    if (rc) return rc;  \
  } while (0)
  // what is over affine experts here is exact, whatever the width from which other calls run as GEMMs
  auto linears = [&](const ornith_linear* const* ws, int n, const void* x, void* const* ys) {
    return ex_affine4 ? linear_exact_multi(ctx, ws, n, x, T, ys) : ornith_linear_matmul_multi(ctx, ws, n, x, T, ys);
  };
  if (ornith_option_fuse_moe() && moe_fused_supported(w)) {
    int rrc = ORNITH_OK;
    // router, up and down as one launch where the shapes are in its family
    if (moe_one_launch(ctx, w, d_x, T, gates, eg, inds, scores, act, d_out, pre, &rrc)) {
      if (rrc) return rrc;
      return ORNITH_OK;
    }
    // gates + shared-expert gate, softmax + top-k, then the two expert kernels
    if (moe_fused_router(ctx, w, d_x, T, gates, eg, &rrc, pre)) {
      if (rrc) return rrc;
    } else {
      if (pre) TRY(ornith_add_rms_norm(ctx, pre->res, pre->y, pre->w, T, H, pre->eps, pre->h_out, pre->normed_out));
      TRY(ornith_linear_matmul(ctx, &w->router, d_x, T, gates));
      TRY(ornith_linear_matmul(ctx, &w->sh_egate, d_x, T, eg));
    }
    // softmax + top-k ride in the head of the up kernel (the reference folds its routing
    // tail the same way, ORNITH_FUSE_MOE_TAIL); E must be one of the wavefront layouts
    const bool topk_in_up = E % 64 == 0 && E <= 1024 && ((E / 64) & (E / 64 - 1)) == 0 && k <= 16;
    if (!topk_in_up) TRY(launch_router(ctx, gates, T, E, k, inds, scores, nullptr, nullptr, nullptr));
    TRY(moe_fused_experts(ctx, w, d_x, T, inds, scores, eg, act, d_out, 3, topk_in_up ? gates : nullptr));
    return ORNITH_OK;
  }
  const bool pair_dense = w->ex_dense && moe_dense_supported(w);
  if (ornith_option_fuse_moe() && (pair_a4 || pair_dense)) {
    // the published artifact's block, and the MTP head's dense one, in three launches: router +
    // shared-expert gate (one launch when their formats match), then the two expert launches of
    // moe_affine4.hip, the softmax + top-k in the head of the first where the expert count allows
    const ornith_linear* in2[2] = {&w->router, &w->sh_egate};
    void* out2[2] = {gates, eg};
    if (pre)  // (falls back to the separate norm where the launch does not cover the shapes)
      TRY(ornith_add_rms_linear_multi(ctx, in2, 2, pre->res, pre->y, pre->w, pre->eps, T, pre->h_out, pre->normed_out, out2));
    else
      TRY(linears(in2, 2, d_x, out2));
    const bool topk_in_up = E % 64 == 0 && E <= 1024 && ((E / 64) & (E / 64 - 1)) == 0 && k <= 16;
    if (!topk_in_up) TRY(launch_router(ctx, gates, T, E, k, inds, scores, nullptr, nullptr, nullptr));
    if (pair_a4)
      TRY(moe_affine4_experts(ctx, w, d_x, T, inds, scores, eg, act, d_out, topk_in_up ? gates : nullptr));
    else
      TRY(moe_dense_experts(ctx, w, d_x, T, inds, scores, eg, act, d_out, topk_in_up ? gates : nullptr));
    return ORNITH_OK;
  }
  {
    // the four projections of the block's input: one launch when their formats allow
    const ornith_linear* in4[4] = {&w->router, &w->sh_gate, &w->sh_up, &w->sh_egate};
    void* out4[4] = {gates, sg, su, eg};
    TRY(linears(in4, 4, d_x, out4));
  }
  TRY(launch_router(ctx, gates, T, E, k, inds, scores, nullptr, lhs_tok, lhs_row));
  if (w->ex_dense) {
    ORN_REQUIRE(w->d_ex_gate && w->d_ex_up && w->d_ex_down, "moe_block: dense expert tensor missing");
    const void* gu[2] = {w->d_ex_gate, w->d_ex_up};
    void* xgu[2] = {xg, xu};
    TRY(dense_gather_mv_multi(ctx, gu, 2, E, I, H, d_x, T, lhs_tok, inds, T * k, xgu));
    // the shared expert's activation and the routed experts' in one launch
    TRY(swiglu_pair(ctx, sg, su, (int64_t)T * SI, sact, xg, xu, (int64_t)T * k * I, act));
    TRY(ornith_linear_matmul(ctx, &w->sh_down, sact, T, sy));
    TRY(ornith_dense_gather_mv(ctx, w->d_ex_down, E, H, I, act, T * k, lhs_row, inds, T * k, y));
  } else if (ex_affine4) {
    // quantized::gather_qmv over the stacked 4-bit affine experts (src/ops/quantized.rs:531-589)
    TRY(ornith_affine4_gather_qmv(ctx, w->ex_gate.d_qs, w->ex_gate.d_scales, w->ex_gate.d_dm, E, I, H, d_x, T,
                                  lhs_tok, inds, T * k, xg));
    TRY(ornith_affine4_gather_qmv(ctx, w->ex_up.d_qs, w->ex_up.d_scales, w->ex_up.d_dm, E, I, H, d_x, T, lhs_tok,
                                  inds, T * k, xu));
    TRY(swiglu_pair(ctx, sg, su, (int64_t)T * SI, sact, xg, xu, (int64_t)T * k * I, act));
    const ornith_linear* const shd = &w->sh_down;
    void* const shy = sy;
    TRY(linears(&shd, 1, sact, &shy));
    TRY(ornith_affine4_gather_qmv(ctx, w->ex_down.d_qs, w->ex_down.d_scales, w->ex_down.d_dm, E, H, I, act, T * k,
                                  lhs_row, inds, T * k, y));
  } else {
    TRY(ornith_kq_gather_qmv(ctx, &w->ex_gate, d_x, ORNITH_BF16, T, lhs_tok, inds, T * k, xg,
                             ORNITH_BF16));
    TRY(ornith_kq_gather_qmv(ctx, &w->ex_up, d_x, ORNITH_BF16, T, lhs_tok, inds, T * k, xu,
                             ORNITH_BF16));
    TRY(swiglu_pair(ctx, sg, su, (int64_t)T * SI, sact, xg, xu, (int64_t)T * k * I, act));
    TRY(ornith_linear_matmul(ctx, &w->sh_down, sact, T, sy));
    TRY(ornith_kq_gather_qmv(ctx, &w->ex_down, act, ORNITH_BF16, T * k, lhs_row, inds, T * k, y,
                             ORNITH_BF16));
  }
  TRY(ornith_moe_combine(ctx, scores, y, eg, sy, T, k, H, w->norm_topk_prob, d_out));
#undef TRY
  return ORNITH_OK;
}

}  // extern "C"

// ornith_add_rms_moe_block with what follows it in the model, if that could ride along (close->done)
int add_rms_moe_block_close(ornith_ctx* ctx, const ornith_moe_weights* w, const PreNorm& pre, int T, void* d_out, MoeClose* close) {
  return moe_block_impl(ctx, w, pre.normed_out, T, d_out, nullptr, nullptr, &pre, true, close);
}

extern "C" {

int ornith_moe_block(ornith_ctx* ctx, const ornith_moe_weights* w, const void* d_x, int T,
                     void* d_out, uint32_t* d_inds_out, void* d_scores_out) {
  return moe_block_impl(ctx, w, d_x, T, d_out, d_inds_out, d_scores_out, nullptr, false);
}

int ornith_add_rms_moe_block(ornith_ctx* ctx, const ornith_moe_weights* w, const void* d_res,
                             const void* d_y, const void* d_wnorm, float eps, int T, void* d_h_out,
                             void* d_normed_out, void* d_out) {
  ORN_REQUIRE(d_res && d_y && d_wnorm && d_h_out && d_normed_out, "add_rms_moe_block: null argument");
  const PreNorm pre{(const bf16_t*)d_res, (const bf16_t*)d_y, (const bf16_t*)d_wnorm, (bf16_t*)d_h_out,
                    (bf16_t*)d_normed_out, eps};
  return moe_block_impl(ctx, w, d_normed_out, T, d_out, nullptr, nullptr, &pre, true);
}

int ornith_selftest_moe_close(ornith_ctx* ctx, const ornith_moe_weights* w, const void* d_res, const void* d_y, const void* d_wnorm,
                              const void* d_wnext, float eps, int T, void* d_h, void* d_normed, void* d_out, void* d_x_out,
                              void* d_next_out, int* done) {
  ORN_REQUIRE(d_res && d_y && d_wnorm && d_wnext && d_h && d_normed && d_x_out && d_next_out && done, "moe_close: null argument");
  const PreNorm pre{(const bf16_t*)d_res, (const bf16_t*)d_y, (const bf16_t*)d_wnorm, (bf16_t*)d_h, (bf16_t*)d_normed, eps};
  MoeClose close{{(const bf16_t*)d_h, nullptr, (const bf16_t*)d_wnext, (bf16_t*)d_x_out, (bf16_t*)d_next_out, eps}};
  const int rc = add_rms_moe_block_close(ctx, w, pre, T, d_out, &close);
  *done = close.done;
  return rc;
}

}  // extern "C"
