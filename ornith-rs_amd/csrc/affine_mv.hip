// Mat-vecs over mlx affine weights (4-bit group 32, 8-bit group 64) at decode widths: up to four
// matrices of one K over the same activation rows in a launch, each row of weights read once for up
// to four activation rows, the layer's residual add + RMS norm in the launch's head.
//
// Replaces quantized::qmv (/root/reference/src/ops/quantized.rs:249-333) where K is 1024, 2048 or
// 4096; other widths keep the row-a-wavefront kernels of linear.hip. The sums are those of
// affine_device.h, so both give the same bits, and a row of an M-row call those of the row alone.
//
// What bounds it: the launch's chain of latencies at projection sizes, vector instructions at the
// output head (2.1 an activation row and weight). So a wavefront has the codes and scales of its
// first rows on their way before anything else (behind the few KB of activations or of the norm's
// inputs, because loads return in issue order), keeps the activations in registers while it walks
// down its rows, and unpacks a row once for all activation rows. One activation row at a time, a row
// of weights a wavefront and a loop over its chunks, the kernels before this one read every weight M
// times with one trip to memory a chunk. us at two activation rows, before -> now: 12288 x 2048 in two
// matrices with the norm 15.9 -> 9.7, a 256-row 8-bit router with the norm and a one-row gate 10.0 -> 4.4,
// 248320 x 2048 180 -> 73 (4.3 TB/s).
#include "affine_device.h"
#include "norm_device.h"
#include "rt.h"

namespace {

struct AffSeg {
  const uint8_t* w;
  const bf16_t *s, *b;
  bf16_t* y;
  int O, first_block, bits;
};

struct AffArgs {
  AffSeg seg[4];
  int nseg;
  const bf16_t* x;  // [Mt, K]
  int Mt;           // activation rows of the call; grid.y takes M at a time
  int iters;        // groups of rows a wavefront walks
  PreNorm pre;
};

// Weight rows of a wavefront's step: as many as make four sums (which fold as one), half of that at
// K = 4096, whose rows hold twice the registers
template <int NC, int M>
constexpr int group_rows() { return M > 2 ? 1 : (NC == 4 ? 2 : 4) / M; }

// One workgroup's rows of one matrix. `issue` asks for what the head of the launch needs, `finish`
// makes the activation rows and gives their addresses.
template <int BITS, int NC, int M, bool ONE, class Issue, class Finish>
__device__ __forceinline__ void aff_rows(const AffSeg& sg, int block, int iters, int m0, int Mt, Issue issue, Finish finish) {
  // (the 8-bit matrices are narrow ones, routers and gates: a row a step)
  constexpr int G = BITS == 8 ? 1 : group_rows<NC, M>(), PF = ONE ? 1 : 2;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int base = (block * 4 + wave) * G * iters;
  const auto L = issue();
  AffRow<BITS, 64, NC> pf[PF][G];
  auto fetch = [&](int it, AffRow<BITS, 64, NC> (&r)[G]) {
#pragma unroll
    for (int g = 0; g < G; ++g) r[g].load(sg.w, sg.s, sg.b, min(base + it * G + g, sg.O - 1), lane);
  };
#pragma unroll
  for (int i = 0; i < PF; ++i) fetch(min(i, iters - 1), pf[i]);
  __builtin_amdgcn_sched_barrier(0);
  const auto X = finish(L);
  for (int it0 = 0; it0 < (ONE ? 1 : iters); it0 += PF) {
#pragma unroll
    for (int i = 0; i < PF; ++i) {
      const int it = it0 + i;
      if (!ONE && it >= iters) break;
      float v[4] = {0.f, 0.f, 0.f, 0.f};  // sum of (row g, activation t) at g * M + t
#pragma unroll
      for (int g = 0; g < G; ++g) {
        float acc[M];
#pragma unroll
        for (int t = 0; t < M; ++t) acc[t] = 0.f;
        pf[i][g].accumulate(X, acc);
#pragma unroll
        for (int t = 0; t < M; ++t) v[g * M + t] = acc[t];
        if (g + 1 < G) pf[i][g + 1].after(acc);
      }
      // (past the end the last group again: loads under a condition would make every use wait for
      // all loads in flight)
      if constexpr (!ONE) fetch(min(it + PF, iters - 1), pf[i]);
      __builtin_amdgcn_sched_barrier(0);
      const float r = dm_wave_sum4(v[0], v[1], v[2], v[3]);
      // lane 0 holds sum 0, lane 16 sum 2, lane 32 sum 1, lane 48 sum 3
      const int k = ((lane >> 5) & 1) | ((lane >> 3) & 2), g = k / M, t = m0 + k - g * M, o = base + it * G + g;
      if ((lane & 15) == 0 && g < G && t < Mt && o < sg.O) sg.y[(size_t)t * sg.O + o] = dm_f2bf(r);
    }
  }
}

// grid (row blocks of all segments, ceil(Mt / M)), 256 threads; NC: K / 1024; ONE: iters is 1
template <int NC, int M, bool PRE, bool ONE>
__global__ __launch_bounds__(256) void affine_mv_kernel(AffArgs a) {
  AffSeg sg = a.seg[0];
#pragma unroll
  for (int i = 1; i < 4; ++i)
    if (i < a.nseg && (int)blockIdx.x >= a.seg[i].first_block) sg = a.seg[i];
  const int block = (int)blockIdx.x - sg.first_block, m0 = blockIdx.y * M, lane = threadIdx.x & 63;
  const bf16_t* xr[M];
#pragma unroll
  for (int t = 0; t < M; ++t) xr[t] = a.x + (size_t)min(m0 + t, a.Mt - 1) * (1024 * NC);
  if constexpr (PRE) {
    __shared__ PreNormLds<M> pn;
    auto issue = [&]() {
      PreNormRegs<M> pg;
      prenorm_issue<M>(a.pre, pg);
      __builtin_amdgcn_sched_barrier(0);
      return pg;
    };
    auto rows = [&](const PreNormRegs<M>& pg) {
      prenorm_finish<M>(a.pre, pg, blockIdx.x == 0, pn);
#pragma unroll
      for (int t = 0; t < M; ++t) xr[t] = &pn.xn[t][0];
    };
    if (sg.bits == 4)
      aff_rows<4, NC, M, ONE>(sg, block, a.iters, m0, a.Mt, issue, [&](const PreNormRegs<M>& pg) {
        rows(pg);
        AffLane<4, 64, NC, M> X;
        X.load(xr, lane);
        return X;
      });
    else
      aff_rows<8, 2 * NC, M, ONE>(sg, block, a.iters, m0, a.Mt, issue, [&](const PreNormRegs<M>& pg) {
        rows(pg);
        AffLane<8, 64, 2 * NC, M> X;
        X.load(xr, lane);
        return X;
      });
  } else {
    auto same = [](const auto& X) { return X; };
    if (sg.bits == 4)
      aff_rows<4, NC, M, ONE>(sg, block, a.iters, m0, a.Mt, [&]() {
        AffLane<4, 64, NC, M> X;
        X.load(xr, lane);
        return X;
      }, same);
    else
      aff_rows<8, 2 * NC, M, ONE>(sg, block, a.iters, m0, a.Mt, [&]() {
        AffLane<8, 64, 2 * NC, M> X;
        X.load(xr, lane);
        return X;
      }, same);
  }
}

template <int NC, int M, bool PRE>
int launch(ornith_ctx* ctx, AffArgs& a) {
  static const int resident = [] {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, affine_mv_kernel<NC, M, PRE, false>, 256, 0) != hipSuccess || n < 1) {
      (void)hipGetLastError();
      n = 2;
    }
    return n;
  }();
  // Groups a wavefront walks: the fewest with which the whole grid is resident at once, counting at
  // most three workgroups a compute unit (a grid the chip does not hold at once runs as two rounds of
  // the same latencies; more workgroups only repeat the activations' conversion), and no more than 8
  // (from there the rows' stream is what counts).
  const int gy = (a.Mt + M - 1) / M;
  const long room = (long)ctx->compute_units * (resident < 3 ? resident : 3);
  int blocks = 0;
  for (a.iters = 1;; ++a.iters) {
    blocks = 0;
    for (int i = 0; i < a.nseg; ++i) {
      const int rows = 4 * (a.seg[i].bits == 8 ? 1 : group_rows<NC, M>()) * a.iters;
      a.seg[i].first_block = blocks;
      blocks += (a.seg[i].O + rows - 1) / rows;
    }
    if (a.iters == 8 || (long)blocks * gy <= room) break;
  }
  if (a.iters == 1)
    hipLaunchKernelGGL((affine_mv_kernel<NC, M, PRE, true>), dim3(blocks, gy), dim3(256), 0, ctx->stream, a);
  else
    hipLaunchKernelGGL((affine_mv_kernel<NC, M, PRE, false>), dim3(blocks, gy), dim3(256), 0, ctx->stream, a);
  ORN_LAUNCH_CHECK("affine_mv_kernel");
  return ORNITH_OK;
}

}  // namespace

// ys[i] = x . ws[i]^T for n affine matrices of one K; with pre, x = rms_norm(pre->res + pre->y) is
// made in the launch (M <= 4, K == 2048). -1 (nothing launched): not covered.
int affine_mv_multi(ornith_ctx* ctx, const ornith_linear* const* ws, int n, const void* d_x, int M, void* const* d_ys,
                    const PreNorm* pre) {
  if (n < 1 || n > 4 || M < 1 || M > 65535) return -1;
  const int K = ws[0]->K;
  if (K != 1024 && K != 2048 && K != 4096) return -1;
  if (pre && (M > 4 || K != kPreN)) return -1;
  // (the norm's own launch, which takes the call then, refuses operands that are not 16-byte aligned)
  if (pre && (((uintptr_t)pre->res | (uintptr_t)pre->y | (uintptr_t)pre->w | (uintptr_t)pre->h_out | (uintptr_t)pre->normed_out) & 15) != 0)
    return -1;
  if (!pre && ((uintptr_t)d_x & 15) != 0) return -1;
  AffArgs a{};
  a.nseg = n;
  a.x = (const bf16_t*)d_x;
  a.Mt = M;
  if (pre) a.pre = *pre;
  for (int i = 0; i < n; ++i) {
    const ornith_linear& w = *ws[i];
    if ((w.mode != ORNITH_LIN_AFFINE4 && w.mode != ORNITH_LIN_AFFINE8) || w.K != K || w.O < 1 || !w.d_w || !w.d_scales ||
        !w.d_biases || !d_ys[i] || ((uintptr_t)w.d_w & 7) != 0)
      return -1;
    a.seg[i] = {(const uint8_t*)w.d_w, (const bf16_t*)w.d_scales, (const bf16_t*)w.d_biases, (bf16_t*)d_ys[i], w.O, 0,
                w.mode == ORNITH_LIN_AFFINE4 ? 4 : 8};
  }
  // Activation rows a workgroup: up to four at K <= 2048, whose lanes keep 32 activations a row in
  // registers, two at 4096; more rows go in equal shares along grid.y.
  const int most = K == 4096 ? 2 : 4, shares = (M + most - 1) / most, m = (M + shares - 1) / shares;
  if (pre) {
    switch (m) {
      case 1: return launch<2, 1, true>(ctx, a);
      case 2: return launch<2, 2, true>(ctx, a);
      case 3: return launch<2, 3, true>(ctx, a);
      default: return launch<2, 4, true>(ctx, a);
    }
  }
#define AFF_M(NC)                                        \
  switch (m) {                                           \
    case 1: return launch<NC, 1, false>(ctx, a);         \
    case 2: return launch<NC, 2, false>(ctx, a);         \
    case 3: return launch<NC, 3, false>(ctx, a);         \
    default: return launch<NC, 4, false>(ctx, a);        \
  }
  if (K == 1024) AFF_M(1)
  if (K == 2048) AFF_M(2)
#undef AFF_M
  return m == 1 ? launch<4, 1, false>(ctx, a) : launch<4, 2, false>(ctx, a);
}
