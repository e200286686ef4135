// The expert half of the MoE block for the two formats whose row dot is one wavefront a row:
// the published artifact's (routed and shared experts in mlx 4-bit affine, group 32,
// /root/reference/src/ops/quantized.rs:311-333,531-589) and the MTP head's (dense bf16 experts,
// /root/reference/src/model/mtp.rs, gather_mm over [E, O, K] tensors). The operator path is
// moe.hip. Two launches that mirror moe_up_kernel / moe_down_kernel
// (moe_fused.hip) in place of five (two gathered mat-vecs, swiglu, the shared expert's down
// projection, the gathered down projection, the combine):
//
// moe_up_affine4:   a wavefront per (token, expert slot | shared, output row): the gate and the
//                   up row over the same activation registers, swiglu -> act. With `gates` the
//                   softmax + top-k of the row's token is made in the head of the launch.
// moe_down_affine4: a workgroup per (token, eight output columns), wavefront j = expert slot j
//                   (the last the shared expert): eight row dots each, met in LDS, then the
//                   block's tail (router weights, bf16 accumulation in slot order, sigmoid-gated
//                   shared expert).
// moe_up_a4, moe_down_a4: the same launches with the same sums for 4-bit rows of 1024, 2048 or 4096 columns
//                   (up) and of 256 or 512 (down), the widths of this model family; other widths and the
//                   dense format take the two above, which cost 1.5 to 4.4 times as much (figures at each).
//
// A 4-bit row dot is affine4_qmv_kernel's (linear.hip), operation for operation: lane l owns the
// 16-code chunks l + 64c in ascending c, one fma chain a chunk in code order beside the plain
// sum of its activations, scale * chain + bias * sum per chunk added to the lane's running
// value, then the 64-lane butterfly; a dense one is dense_row_dot (linear_device.h), the
// function the operator path's kernels call. So the two launches give the bits of the operator
// path and of the oracle (oracle/orc_moe.c).
#include "affine_device.h"
#include "linear_device.h"
#include "moe_device.h"
#include "rt.h"

namespace {

constexpr int kA4MaxK = 8;  // routed experts a token the down kernel's workgroup holds

struct A4Mat {
  const uint8_t* w;      // [rows, K/2]
  const bf16_t* scales;  // [rows, K/32]
  const bf16_t* biases;  // [rows, K/32]
};

// 16 activations of chunk j as floats, and their sum in code order
struct A4X {
  float v[16];
  float sum;
  __device__ __forceinline__ void load(const bf16_t* xr, int j) {
    const uint4 xa = *reinterpret_cast<const uint4*>(xr + 16 * j);
    const uint4 xb = *reinterpret_cast<const uint4*>(xr + 16 * j + 8);
    const uint32_t wds[8] = {xa.x, xa.y, xa.z, xa.w, xb.x, xb.y, xb.z, xb.w};
    sum = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      v[2 * i] = dm_bf2f_lo(wds[i]);
      v[2 * i + 1] = dm_bf2f_hi(wds[i]);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) sum = sum + v[i];
  }
};

// one chunk's contribution: scale * sum_i x_i q_i + bias * sum_i x_i
__device__ __forceinline__ float a4_chunk(const A4Mat& m, size_t row, int K, int j, const A4X& x) {
  const uint2 q = *reinterpret_cast<const uint2*>(m.w + row * (K / 2) + 8 * j);
  const uint32_t qw[2] = {q.x, q.y};
  float acc = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const float qf = (float)((qw[i >> 3] >> (4 * (i & 7))) & 0xfu);
    acc = dm_fma(x.v[i], qf, acc);
  }
  const float s = dm_bf2f(m.scales[row * (K / 32) + (j >> 1)]), b = dm_bf2f(m.biases[row * (K / 32) + (j >> 1)]);
  float p = s * acc;
  return dm_fma(x.sum, b, p);
}

// The two formats behind one pair of kernels: a matrix handle, the gate and up rows' dots over
// one activation row, and NC rows' dots of one matrix.
struct FmtA4 {
  using Mat = A4Mat;
  static __device__ __forceinline__ void dot2(const Mat& wg, const Mat& wu, size_t row, int K, const bf16_t* xr,
                                              int lane, float& g, float& u) {
    float ag = 0.f, au = 0.f;
    for (int j = lane; j < K / 16; j += 64) {
      A4X x;
      x.load(xr, j);
      ag = ag + a4_chunk(wg, row, K, j, x);
      au = au + a4_chunk(wu, row, K, j, x);
    }
    g = dm_wave_sum<64>(ag);
    u = dm_wave_sum<64>(au);
  }
  template <int NC>
  static __device__ __forceinline__ void dotn(const Mat& w, size_t row0, int c0, int O, int K, const bf16_t* xr,
                                              int lane, float (&v)[NC]) {
    float acc[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[c] = 0.f;
    for (int jj = lane; jj < K / 16; jj += 64) {
      A4X x;
      x.load(xr, jj);
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int o = c0 + c < O ? c0 + c : O - 1;
        acc[c] = acc[c] + a4_chunk(w, row0 + o, K, jj, x);
      }
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) v[c] = dm_wave_sum<64>(acc[c]);
  }
};

struct DenseMat {
  const bf16_t* w;  // [rows, K]
};
struct FmtDense {
  using Mat = DenseMat;
  static __device__ __forceinline__ void dot2(const Mat& wg, const Mat& wu, size_t row, int K, const bf16_t* xr,
                                              int lane, float& g, float& u) {
    const bf16_t* const rows[2] = {wg.w + row * K, wu.w + row * K};
    float v[2];
    dense_rows_dot<2, 4>(rows, xr, K, lane, v);
    g = v[0];
    u = v[1];
  }
  template <int NC>
  static __device__ __forceinline__ void dotn(const Mat& w, size_t row0, int c0, int O, int K, const bf16_t* xr,
                                              int lane, float (&v)[NC]) {
    const bf16_t* rows[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int o = c0 + c < O ? c0 + c : O - 1;
      rows[c] = w.w + (row0 + o) * K;
    }
    dense_rows_dot<NC, 1>(rows, xr, K, lane, v);
  }
};

template <class F>
struct A4UpArgs {
  typename F::Mat gate, up;    // routed [E * I, K]
  typename F::Mat sgate, sup;  // shared [I, K]
  const bf16_t* x;       // [T, K]
  const uint32_t* inds;  // [T*k], read unless gates is given
  bf16_t* act;           // [T*k + T, I]
  int T, k, E, I, K;
  const bf16_t* gates;   // [T, E] or null
  uint32_t* inds_out;    // [T*k]
  bf16_t* scores_out;    // [T*k]
};

// What row blockIdx.y of an up launch works on: its token, the first weight row of its expert and
// the two matrices. With ROUTE softmax + top-k of the row's token are made here.
template <class F>
struct A4UpRow {
  int token;
  size_t row0;
  typename F::Mat wg, wu;
};
template <class F, bool ROUTE>
__device__ __forceinline__ A4UpRow<F> a4_up_row(const A4UpArgs<F>& a, int lane, int wave) {
  const int r = blockIdx.y, routed = a.T * a.k;
  A4UpRow<F> u;
  if (r < routed) {
    u.token = r / a.k;
    uint32_t e;
    if constexpr (ROUTE) {
      __shared__ uint32_t s_inds[16];
      __shared__ bf16_t s_scores[16];
      if (wave == 0) {
        const bf16_t* g = a.gates + (size_t)u.token * a.E;
        switch (a.E / 64) {
          case 1: router_topk_wave<1>(g, a.k, s_inds, s_scores, nullptr, lane); break;
          case 2: router_topk_wave<2>(g, a.k, s_inds, s_scores, nullptr, lane); break;
          case 4: router_topk_wave<4>(g, a.k, s_inds, s_scores, nullptr, lane); break;
          case 8: router_topk_wave<8>(g, a.k, s_inds, s_scores, nullptr, lane); break;
          default: router_topk_wave<16>(g, a.k, s_inds, s_scores, nullptr, lane); break;
        }
      }
      __syncthreads();
      e = s_inds[r - u.token * a.k];
      if (blockIdx.x == 0 && r == u.token * a.k && (int)threadIdx.x < a.k) {
        a.inds_out[r + threadIdx.x] = s_inds[threadIdx.x];
        a.scores_out[r + threadIdx.x] = s_scores[threadIdx.x];
      }
    } else {
      e = a.inds[r];
    }
    u.row0 = (size_t)min(e, (uint32_t)(a.E - 1)) * a.I;
    u.wg = a.gate;
    u.wu = a.up;
  } else {
    u.token = r - routed;
    u.row0 = 0;
    u.wg = a.sgate;
    u.wu = a.sup;
  }
  return u;
}

// grid (ceil(I / 4), T*k + T), 256 threads: a wavefront an output row
template <class F, bool ROUTE>
__global__ __launch_bounds__(256) void moe_up_affine4_kernel(A4UpArgs<F> a) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = blockIdx.y;
  const A4UpRow<F> u = a4_up_row<F, ROUTE>(a, lane, wave);
  const int o = blockIdx.x * 4 + wave;
  if (o >= a.I) return;
  const bf16_t* xr = a.x + (size_t)u.token * a.K;
  float gs, us;
  F::dot2(u.wg, u.wu, u.row0 + o, a.K, xr, lane, gs, us);
  if (lane == 0) a.act[(size_t)r * a.I + o] = swiglu_bf16(gs, us);
}

// The same for 4-bit rows of K = 1024 NC: two intermediate rows a wavefront, the codes and scales of
// their gate and up rows asked for together and the four sums folded as one. What bounds it is the
// chain gates -> top-k -> rows -> sums; the kernel above, which every other width takes, adds a trip
// to memory for every 1024 columns of a row and unpacks with three instructions a code where this
// one needs one and a half. LOOPS as in moe_up_kernel (moe_fused.hip): the next two rows asked for ahead
// of the arithmetic of the present ones, once the grid is more than the chip holds. us at T = 1 / 2, K = 2048, I = 512: 11.3 / 16.6 -> 7.3 / 10.2
// The routing is always made in its head: the block has it nowhere else for the expert counts it takes.
// grid (ceil(I / (8 LOOPS)), T*k + T), 256 threads
template <int NC, int LOOPS>
__global__ __launch_bounds__(256) void moe_up_a4_kernel(A4UpArgs<FmtA4> a) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = blockIdx.y;
  const A4UpRow<FmtA4> u = a4_up_row<FmtA4, true>(a, lane, wave);
  const int base0 = (blockIdx.x * 4 + wave) * 2 * LOOPS;
  constexpr int SETS = LOOPS > 1 ? 2 : 1;
  AffRow<4, 64, NC> rows[SETS][4];  // gate 0, up 0, gate 1, up 1
  auto fetch = [&](int l) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const size_t row = u.row0 + min(base0 + 2 * l + i, a.I - 1);
      rows[l % SETS][2 * i].load(u.wg.w, u.wg.scales, u.wg.biases, row, lane);
      rows[l % SETS][2 * i + 1].load(u.wu.w, u.wu.scales, u.wu.biases, row, lane);
    }
  };
  fetch(0);
  __builtin_amdgcn_sched_barrier(0);
  AffLane<4, 64, NC, 1> L;
  const bf16_t* xr[1] = {a.x + (size_t)u.token * a.K};
  L.load(xr, lane);
#pragma unroll
  for (int l = 0; l < LOOPS; ++l) {
    if (l + 1 < LOOPS) {
      fetch(l + 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float acc[1] = {0.f};
      rows[l % SETS][i].accumulate(L, acc);
      v[i] = acc[0];
      if (LOOPS > 1 && i < 3) rows[l % SETS][i + 1].after(acc);
    }
    // lanes [0,16): gate row 0, [32,48): up row 0, [16,32): gate row 1, [48,64): up row 1
    const float red = dm_wave_sum4(v[0], v[1], v[2], v[3]);
    float gs, us;
    dm_row_swap<32>(red, gs, us);
    const int o = base0 + 2 * l + ((lane >> 4) & 1);
    if ((lane & 47) == 0 && o < a.I) a.act[(size_t)r * a.I + o] = swiglu_bf16(gs, us);
  }
}

template <class F>
struct A4DownArgs {
  typename F::Mat down;   // routed [E * H, I]
  typename F::Mat sdown;  // shared [H, I]
  const bf16_t* act;     // [T*k + T, I]
  const uint32_t* inds;  // [T*k]
  const bf16_t* scores;  // [T*k]
  const bf16_t* egate;   // [T]
  bf16_t* out;           // [T, H]
  int T, k, E, H, I, normalize;
};

// the router weights of a token, from its scores (one a lane): denom = ((0+s0)+s1)..., w_j = bf16(s_j / denom)
__device__ __forceinline__ void a4_combine_weights(uint16_t score_bits, uint16_t egate_bits, int k, int normalize, int lane,
                                                   float* wj, float* gsig) {
  float denom = 0.f;
  if (normalize) {
#pragma unroll
    for (int i = 0; i < kA4MaxK; ++i)
      if (i < k) denom = dm_rb(dm_bf2f((bf16_t)__builtin_amdgcn_readlane((int)score_bits, i)) + denom);
  }
  if (lane < k) wj[lane] = normalize ? dm_rb(dm_bf2f(score_bits) / denom) : dm_bf2f(score_bits);
  if (lane == 0) *gsig = dm_sigmoid_bf16(dm_bf2f(egate_bits));
}
// one output column of a token: y[i * ld] the experts' sums in slot order, the shared one last
__device__ __forceinline__ bf16_t a4_combine(const float* y, int ld, const float* wj, float gsig, int k) {
  float s = 0.f;
  for (int i = 0; i < k; ++i) {
    const float weighted = dm_rb(y[i * ld] * wj[i]);
    s = dm_rb(weighted + s);
  }
  const float gated = dm_rb(gsig * y[k * ld]);
  return dm_f2bf(s + gated);
}

constexpr int kA4Cols = 8;

// grid (ceil(H / 8), T), 64 * (k + 1) threads
template <class F>
__global__ __launch_bounds__(64 * (kA4MaxK + 1)) void moe_down_affine4_kernel(A4DownArgs<F> a) {
  const int lane = threadIdx.x & 63, j = threadIdx.x >> 6;  // j: expert slot, k = shared
  const int t = blockIdx.y, k = a.k, c0 = blockIdx.x * kA4Cols;
  __shared__ float yl[kA4MaxK + 1][kA4Cols];
  __shared__ float wj[kA4MaxK];
  __shared__ float gsig;
  const bool shared = j == k;
  const int arow = shared ? a.T * k + t : t * k + j;
  const typename F::Mat w = shared ? a.sdown : a.down;
  const size_t row0 = shared ? 0 : (size_t)min(a.inds[t * k + j], (uint32_t)(a.E - 1)) * a.H;
  // the token's router scores (lane i < k holds score i) and shared-expert gate are asked for
  // ahead of the rows and turned into the combine weights once the rows' sums are made: a
  // loop of loads here, one score a trip to memory, held wavefront 0's rows back by all of them
  const uint16_t score_bits = a.scores[(size_t)t * k + (lane < k ? lane : 0)];
  const uint16_t egate_bits = a.egate[t];
  const bf16_t* xr = a.act + (size_t)arow * a.I;
  float v[kA4Cols];
  F::template dotn<kA4Cols>(w, row0, c0, a.H, a.I, xr, lane, v);
  if (j == 0) a4_combine_weights(score_bits, egate_bits, k, a.normalize, lane, wj, &gsig);
#pragma unroll
  for (int c = 0; c < kA4Cols; ++c)
    if (lane == 0) yl[j][c] = dm_rb(v[c]);  // expert outputs are bf16 in the operator path
  __syncthreads();
  const int col = threadIdx.x;
  if (col < kA4Cols && c0 + col < a.H) a.out[(size_t)t * a.H + c0 + col] = a4_combine(&yl[0][col], kA4Cols, wj, gsig, k);
}

// The same for 4-bit rows of I = 16 LPR columns: 64 / LPR output columns a wavefront pass (32 lanes
// are a row of 512: the kernel above left the other half of its wavefronts idle and asked for a row
// after it had worked off the one before), ITERS passes asked for at once. At 32 columns a workgroup
// the shared expert's passes go over four wavefronts, so that the four SIMDs carry the same number.
// us at T = 1 / 2, I = 512, H = 2048: 14.0 / 25.5 -> 4.3 / 5.8
// grid (ceil(H / COLS), T), 64 * (k + 1) threads, 64 * (k + 4) at 32 columns
constexpr int a4_shared_waves(int cols) { return cols >= 32 ? 4 : 1; }
template <int LPR, int ITERS>
__global__ __launch_bounds__(64 * (kA4MaxK + a4_shared_waves(64 / LPR * ITERS))) void moe_down_a4_kernel(A4DownArgs<FmtA4> a) {
  constexpr int RPW = 64 / LPR, COLS = RPW * ITERS, SW = a4_shared_waves(COLS), SHARE = ITERS / SW;
  const int lane = threadIdx.x & 63, j = threadIdx.x >> 6;  // j < k: expert slot, else the shared expert
  const int slot = lane / LPR, c = lane % LPR;
  const int t = blockIdx.y, k = a.k, c0 = blockIdx.x * COLS;
  __shared__ float yl[kA4MaxK + 1][COLS];
  __shared__ float wj[kA4MaxK];
  __shared__ float gsig;
  const bool shared = j >= k;
  const int it0 = shared ? (j - k) * SHARE : 0, its = shared ? SHARE : ITERS;
  static_assert(SHARE <= 16, "a shared wavefront's passes fit its registers");
  const FmtA4::Mat w = shared ? a.sdown : a.down;
  const size_t row0 = shared ? 0 : (size_t)min(a.inds[t * k + j], (uint32_t)(a.E - 1)) * a.H;
  // what is small and cached first: loads return in issue order
  AffLane<4, LPR, 1, 1> L;
  const bf16_t* xr[1] = {a.act + (size_t)(shared ? a.T * k + t : t * k + j) * a.I};
  L.load(xr, c);
  const uint16_t score_bits = a.scores[(size_t)t * k + (lane < k ? lane : 0)];
  const uint16_t egate_bits = a.egate[t];
  __builtin_amdgcn_sched_barrier(0);
  constexpr int PF = ITERS < 16 ? ITERS : 16;
  AffRow<4, LPR, 1> rr[PF];
  auto fetch = [&](int i) { rr[i % PF].load(w.w, w.scales, w.biases, row0 + min(c0 + (it0 + i) * RPW + slot, a.H - 1), c); };
#pragma unroll
  for (int i = 0; i < PF; ++i)
    if (SW == 1 || i < its) fetch(i);
  __builtin_amdgcn_sched_barrier(0);
  if (j == 0) a4_combine_weights(score_bits, egate_bits, k, a.normalize, lane, wj, &gsig);
  auto pass = [&](int i) {
    float acc[1] = {0.f};
    rr[i % PF].accumulate(L, acc);
    const float v = dm_wave_sum<LPR>(acc[0]);
    if (c == 0) yl[shared ? k : j][(it0 + i) * RPW + slot] = dm_rb(v);  // expert outputs are bf16 in the operator path
  };
  if (SW > 1 && shared) {
#pragma unroll
    for (int i = 0; i < SHARE; ++i) pass(i);
  } else {
#pragma unroll
    for (int i = 0; i < ITERS; ++i) {
      pass(i);
      if (i + PF < ITERS) fetch(i + PF);
    }
  }
  __syncthreads();
  const int col = threadIdx.x;
  if (col < COLS && c0 + col < a.H) a.out[(size_t)t * a.H + c0 + col] = a4_combine(&yl[0][col], COLS, wj, gsig, k);
}

A4Mat mat_of(const ornith_kmatrix& m) {
  return A4Mat{(const uint8_t*)m.d_qs, (const bf16_t*)m.d_scales, (const bf16_t*)m.d_dm};
}
A4Mat mat_of(const ornith_linear& l) {
  return A4Mat{(const uint8_t*)l.d_w, (const bf16_t*)l.d_scales, (const bf16_t*)l.d_biases};
}

}  // namespace

// Whether the two launches cover this block: routed and shared experts all 4-bit affine
// group 32, shapes that chain, at most 8 routed experts a token.
bool moe_affine4_supported(const ornith_moe_weights* w) {
  if (w->ex_dense) return false;
  if (w->ex_gate.kind != ORNITH_AFFINE4_G32 || w->ex_up.kind != ORNITH_AFFINE4_G32 ||
      w->ex_down.kind != ORNITH_AFFINE4_G32)
    return false;
  const ornith_linear* sh[3] = {&w->sh_gate, &w->sh_up, &w->sh_down};
  for (auto* l : sh)
    if (l->mode != ORNITH_LIN_AFFINE4) return false;
  if (w->sh_gate.O != w->ex_gate.O || w->sh_up.O != w->ex_gate.O || w->sh_down.K != w->ex_gate.O) return false;
  if (w->top_k < 1 || w->top_k > kA4MaxK) return false;
  return w->ex_gate.K % 32 == 0 && w->ex_gate.O % 32 == 0;
}

namespace {

// the 4-bit kernels of fixed width; false: another format or width
template <class F>
bool launch_up_a4(ornith_ctx*, const A4UpArgs<F>&) { return false; }
bool launch_up_a4(ornith_ctx* ctx, const A4UpArgs<FmtA4>& u) {
  if (!u.gates) return false;
  const int rows_y = u.T * u.k + u.T, nc = u.K % 1024 == 0 ? u.K / 1024 : 0;
  const long one = (long)((u.I + 7) / 8) * rows_y;
  const int loops = one <= 5L * ctx->compute_units ? 1 : one <= 9L * ctx->compute_units ? 2 : 4;
  const dim3 grid((u.I + 8 * loops - 1) / (8 * loops), rows_y);
#define UP_GO(NC, LOOPS) hipLaunchKernelGGL((moe_up_a4_kernel<NC, LOOPS>), grid, dim3(256), 0, ctx->stream, u)
#define UP_NC(NC)                   \
  if (loops == 1) UP_GO(NC, 1);      \
  else if (loops == 2) UP_GO(NC, 2); \
  else UP_GO(NC, 4);                 \
  return true;
  switch (nc) {
    case 1: UP_NC(1)
    case 2: UP_NC(2)
    case 4: UP_NC(4)
    default: return false;
  }
#undef UP_GO
#undef UP_NC
}
template <class F>
bool launch_down_a4(ornith_ctx*, const A4DownArgs<F>&) { return false; }
bool launch_down_a4(ornith_ctx* ctx, const A4DownArgs<FmtA4>& d) {
  // columns a workgroup: 8 while that is no more than two workgroups a compute unit, then 16, then 32
  const int g8 = (d.H + 7) / 8 * d.T, cu = ctx->compute_units;
  // (and 64, half of them in registers at any time, once 32 are more workgroups than the chip holds)
  const int cols = g8 > 4 * cu ? 64 : g8 >= 3 * cu ? 32 : g8 >= 2 * cu ? 16 : 8;
  const dim3 grid((d.H + cols - 1) / cols, d.T), block(64 * (d.k + a4_shared_waves(cols)));
#define DOWN_LPR(LPR)                                                                                              \
  if (cols == 8)                                                                                                   \
    hipLaunchKernelGGL((moe_down_a4_kernel<LPR, 8 * LPR / 64>), grid, block, 0, ctx->stream, d);                   \
  else if (cols == 16)                                                                                             \
    hipLaunchKernelGGL((moe_down_a4_kernel<LPR, 16 * LPR / 64>), grid, block, 0, ctx->stream, d);                  \
  else if (cols == 32) \
    hipLaunchKernelGGL((moe_down_a4_kernel<LPR, 32 * LPR / 64>), grid, block, 0, ctx->stream, d);                  \
  else \
    hipLaunchKernelGGL((moe_down_a4_kernel<LPR, 64 * LPR / 64>), grid, block, 0, ctx->stream, d);                  \
  return true;
  switch (d.I) {
    case 256: DOWN_LPR(16)
    case 512: DOWN_LPR(32)
    default: return false;
  }
#undef DOWN_LPR
}

template <class F>
int launch_pair(ornith_ctx* ctx, const ornith_moe_weights* w, const typename F::Mat (&m)[6], const void* d_x, int T,
                const uint32_t* d_inds, const void* d_scores, const void* d_egate, void* d_act, void* d_out,
                const void* d_gates) {
  const int E = w->router.O, H = w->router.K, I = w->sh_gate.O, k = w->top_k;
  A4UpArgs<F> u{};
  u.gate = m[0];
  u.up = m[1];
  u.sgate = m[2];
  u.sup = m[3];
  u.x = (const bf16_t*)d_x;
  u.inds = d_inds;
  u.act = (bf16_t*)d_act;
  u.T = T;
  u.k = k;
  u.E = E;
  u.I = I;
  u.K = H;
  u.gates = (const bf16_t*)d_gates;
  u.inds_out = const_cast<uint32_t*>(d_inds);
  u.scores_out = (bf16_t*)const_cast<void*>(d_scores);
  const dim3 ugrid((I + 3) / 4, T * k + T);
  if (launch_up_a4(ctx, u)) {
  } else if (d_gates)
    hipLaunchKernelGGL((moe_up_affine4_kernel<F, true>), ugrid, dim3(256), 0, ctx->stream, u);
  else
    hipLaunchKernelGGL((moe_up_affine4_kernel<F, false>), ugrid, dim3(256), 0, ctx->stream, u);
  ORN_LAUNCH_CHECK("moe_up_affine4_kernel");
  A4DownArgs<F> d{};
  d.down = m[4];
  d.sdown = m[5];
  d.act = (const bf16_t*)d_act;
  d.inds = d_inds;
  d.scores = (const bf16_t*)d_scores;
  d.egate = (const bf16_t*)d_egate;
  d.out = (bf16_t*)d_out;
  d.T = T;
  d.k = k;
  d.E = E;
  d.H = H;
  d.I = I;
  d.normalize = w->norm_topk_prob;
  if (!launch_down_a4(ctx, d)) hipLaunchKernelGGL(moe_down_affine4_kernel<F>, dim3((H + kA4Cols - 1) / kA4Cols, T), dim3(64 * (k + 1)), 0,
                     ctx->stream, d);
  ORN_LAUNCH_CHECK("moe_down_affine4_kernel");
  return ORNITH_OK;
}

}  // namespace

// act: scratch bf16 [(T*k + T), I]. With d_gates the up launch makes the routing and stores it
// to d_inds / d_scores (which then are outputs).
int moe_affine4_experts(ornith_ctx* ctx, const ornith_moe_weights* w, const void* d_x, int T, const uint32_t* d_inds,
                        const void* d_scores, const void* d_egate, void* d_act, void* d_out, const void* d_gates) {
  const A4Mat m[6] = {mat_of(w->ex_gate), mat_of(w->ex_up), mat_of(w->sh_gate),
                      mat_of(w->sh_up),   mat_of(w->ex_down), mat_of(w->sh_down)};
  return launch_pair<FmtA4>(ctx, w, m, d_x, T, d_inds, d_scores, d_egate, d_act, d_out, d_gates);
}

// The same two launches for dense bf16 experts (the MTP head's block): routed tensors [E, O, K]
// and dense shared-expert linears.
bool moe_dense_supported(const ornith_moe_weights* w) {
  if (!w->ex_dense || !w->d_ex_gate || !w->d_ex_up || !w->d_ex_down) return false;
  const ornith_linear* sh[3] = {&w->sh_gate, &w->sh_up, &w->sh_down};
  for (auto* l : sh)
    if (l->mode != ORNITH_LIN_DENSE || !l->d_w) return false;
  if (w->sh_up.O != w->sh_gate.O || w->sh_down.K != w->sh_gate.O || w->sh_gate.K != w->router.K ||
      w->sh_down.O != w->router.K)
    return false;
  if (w->top_k < 1 || w->top_k > kA4MaxK) return false;
  return w->router.K % 8 == 0 && w->sh_gate.O % 8 == 0;
}

int moe_dense_experts(ornith_ctx* ctx, const ornith_moe_weights* w, const void* d_x, int T, const uint32_t* d_inds,
                      const void* d_scores, const void* d_egate, void* d_act, void* d_out, const void* d_gates) {
  const DenseMat m[6] = {{(const bf16_t*)w->d_ex_gate}, {(const bf16_t*)w->d_ex_up},   {(const bf16_t*)w->sh_gate.d_w},
                         {(const bf16_t*)w->sh_up.d_w}, {(const bf16_t*)w->d_ex_down}, {(const bf16_t*)w->sh_down.d_w}};
  return launch_pair<FmtDense>(ctx, w, m, d_x, T, d_inds, d_scores, d_egate, d_act, d_out, d_gates);
}
