// Arguments and launch sizing of the k-quant mat-vecs (kquant.hip, kquant_rows.hip).
#pragma once

#include "norm_device.h"
#include "rt.h"

constexpr int kMaxSeg = 4;

struct KqSeg {
  const uint8_t* qs;
  const uint8_t* scales;
  const uint16_t* dm;
  void* y;
  int O;
  int first_block;
};

struct KqArgs {
  KqSeg seg[kMaxSeg];
  int nseg;
  const void* x;
  const uint32_t* lhs;  // gather only
  const uint32_t* rhs;  // gather only
  int K;
  int E, x_rows;  // gather: bounds for rhs / lhs (out-of-range ids are clamped); x_rows: activation rows
  int iters;      // row iterations per wavefront
  int y_bf16;     // 1: round outputs to bf16, 0: fp32
  PreNorm pre;    // PRE kernels: the activations are rms_norm(res + y) computed by every workgroup
};

// fills first_block for every segment and returns the grid width
template <int LPR, int KS>
int layout_segments(KqArgs& a) {
  constexpr int RPW = 64 / LPR, WPB = 4 / KS;
  const int rows_per_block = RPW * WPB * a.iters;
  int blocks = 0;
  for (int s = 0; s < a.nseg; ++s) {
    a.seg[s].first_block = blocks;
    blocks += (a.seg[s].O + rows_per_block - 1) / rows_per_block;
  }
  return blocks;
}

// Workgroups of a kernel that one compute unit holds at once (its registers and LDS decide:
// from five for one Q4_K activation row down to one for three or four Q6_K rows, whose lanes
// keep 64 activations a row in registers). Asked of the runtime once per kernel.
template <typename Kernel>
int resident_workgroups(Kernel kernel) {
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, 256, 0) != hipSuccess || n < 1) {
    (void)hipGetLastError();
    n = 2;
  }
  return n;
}

// Rows each wavefront walks when the caller leaves it open (a.iters == 0): the fewest with
// which the whole grid is resident at once, counting at most three workgroups a compute unit.
// The kernels are bound by latency and vector-ALU issue, not by HBM: a grid larger than the
// chip holds runs as two rounds of the same chain of latencies (a 9216 x 2048 Q6_K projection
// of two rows: 9.9 us as 1152 workgroups where 512 fit, 8.6 us as 384; one workgroup too many
// costs the same second round: 8192 + 4096 Q4_K rows of four activation rows take 19.0 us as
// 342 + 171 workgroups where 512 fit, 15.8 us as 384), while rows beyond that only lengthen the
// one round; and beyond three workgroups a compute unit the activations' conversion (and a norm
// made in the head) is repeated for nothing. A grid that does not fit with 8 rows a wavefront goes on
// to 32 where several activation rows make the arithmetic the larger part (248320 rows of four
// activation rows 181 -> 165 us, 12288 rows of two groups of four 20.5 -> 18.3), but not for one,
// which is a stream of weights that more workgroups keep fuller (60 us against 67).
template <int LPR, int KS, int M>
int auto_iters(const ornith_ctx* ctx, const KqArgs& a, int grid_y, int resident, int most = 3) {
  constexpr int cap = M > 1 ? 32 : 8;
  constexpr int rows_per_pass = (64 / LPR) * (4 / KS);
  const long room = (long)ctx->compute_units * (resident < most ? resident : most);
  for (int iters = 1; iters < cap; ++iters) {
    long blocks = 0;
    for (int s = 0; s < a.nseg; ++s) blocks += (a.seg[s].O + rows_per_pass * iters - 1) / (rows_per_pass * iters);
    if (blocks * grid_y <= room) return iters;
  }
  return cap;
}

// kquant_rows.hip: the form on the matrix cores
bool kq_rows_suits(const KqArgs& a);
int kq_rows(ornith_ctx* ctx, KqArgs& a, int kind, bool x_f32);
