// The GEMM of long prompts over k-quants (kq_mm_own.hip): what the dispatch of kq_mm.hip fills in and calls.
#pragma once

#include "dmath.h"
#include "rt.h"

struct OwnMat {
  const uint8_t *qs, *scales, *dm;
  bf16_t* y;
  int O, kind;
  int t0;  // plain form: first column tile of the launch that is this matrix's
};

struct OwnArgs {
  OwnMat m[4];  // plain: up to four matrices of one K, of either kind; gathered: the experts' stack
  int n;
  const bf16_t* x;
  int M, K;
  bool halves;  // plain form: the matrices are of kq_mm_own_halves
  int tile_rows, row_tiles, col_tiles;  // set by kq_mm_own
  // gathered form: tiles of up to kOwnRows pairs of an expert-sorted list
  const uint32_t *pair, *tile_expert, *tile_start, *tile_count, *n_tiles;
  int tiles_max, up_div;
  const uint32_t* expert_at;  // over a plan of lower tiles: [E] where an expert's pairs begin; else null
  int E;
  uint32_t up_magic;  // dm_div_magic(up_div)
};

constexpr int kOwnRows = 256, kOwnCols = 256;  // a workgroup's tile (in halves of K, and of a thin launch, 128 x 128)

// alignment and reach: x of `rows` rows, any K % 256 == 0
bool kq_mm_own_ok(const ornith_kmatrix& w, const void* x, size_t rows);
// ... and M rows are many enough, whatever shares the launch (and the option gemm_duo is on); the few-row kernels come first
bool kq_mm_own_suits(const ornith_kmatrix& w, const void* x, int M);
// ... and then whether its sums are taken in two halves of K
bool kq_mm_own_halves(const ornith_kmatrix& w, int M);
// whether a plain launch of whole sums over K takes tiles of 128 x 128 (a.m[].O, n, M, K), on a device of that many compute units: the sums are the same
bool kq_mm_own_thin(const OwnArgs& a, int units);
// ... and a gathered one, by its experts' columns and the pairs of them all
bool kq_mm_own_thin_experts(int O, int E, int pairs, int units);
// kq_mm.hip: the form that kq_gather_matmul takes, as ornith_selftest_gather_form gives it
int kq_gather_form(const ornith_kmatrix& w, const void* d_x, int pairs, int top_k, bool is_up, const void* d_y, int units);
OwnMat kq_mm_own_mat(const ornith_kmatrix& w, void* y);
int kq_mm_own(ornith_ctx* ctx, OwnArgs& a, bool gather);
