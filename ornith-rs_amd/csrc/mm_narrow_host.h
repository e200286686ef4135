// Host side of the few-row GEMM: what the dispatches of linear.hip, kq_mm.hip and moe.hip ask and
// call, and the kernels of one weight family.
#pragma once

#include <algorithm>

#include "mm_narrow.h"

namespace nmm {

// Rows up to which a k-quant projection takes these kernels; more go to the own-column kernel (kq_mm_own.hip, us, here / there). One matrix at a time,
// never by what shares its launch: a matrix gives the same bits alone and in company.
// More than 512 columns: up to 2^20 outputs, about where these kernels' 64-row tiles no longer are one a compute unit (Q4_K x 2048: 1536 columns at 600 / 800 rows
// 13 / 14, 18 / 14, 2048 at 400 / 513 12 / 13, 15 / 14, 3072 at 300 / 400 13 / 16, 18 / 16; x 4096: 2048 at 513 / 600 24 / 24, 30 / 25; Q6_K x 4096: 2048 at 400 /
// 600 25 / 28, 37 / 30), of fewer than 1820 columns 576 rows, of fewer than 910 2^19 outputs: one of those alone is no faster there up to 2^20 either, two
// together are (Q4_K x 4096: 768 at 600 / 800 16 / 24, 24 / 24, 1024 at 513 / 600 / 800 17 / 24, 23 / 24, 22 / 24, two of them at 513 / 700 24 / 24, 30 / 24).
// From 4096 columns on, which come with others as wide, Q4_K 128 rows (8192 + 4096 x 2048 at 100 / 129 rows 18 / 18, 25 / 18), Q6_K 192 (8192 + 512 + 512
// x 2048, of which the narrow ones then run by themselves, at 192 / 200 23 / 24, 35 / 25).
// Up to 512 columns, which rarely come alone, 1024 and of Q4_K 1536; up to 256, a handful of workgroups there, 2560 (256 x 2048 at 1200 / 2000 rows 13 / 15,
// 18 / 15). Below K = 2048 1024 rows up to 2048 columns (264 x 512 at 1025 / 2000 5 / 6, 7 / 6; 2048 x 1024 at 400 / 600 9 / 10, 12 / 10, with two of 512 columns, which
// then run by themselves, at 513 12 / 16).
constexpr int kNarrowOutputs = 1 << 20, kNarrowRows = 192, kNarrowRowsQ4K = 128, kNarrowRowsMid = 576, kNarrowRowsSlim = 1024, kNarrowRowsSlimQ4K = 1536,
              kNarrowRowsSlimmest = 2560;
inline int kq_rows(bool q4, int O, int K) {
  if (O >= 4096) return q4 ? kNarrowRowsQ4K : kNarrowRows;
  if (O > 2048 || (O > 512 && K >= 2048)) return std::min(kNarrowOutputs / O, std::max(kNarrowOutputs / 2 / O, kNarrowRowsMid));
  return K < 2048 ? kNarrowRowsSlim : O <= 256 ? kNarrowRowsSlimmest : q4 && O <= 512 ? kNarrowRowsSlimQ4K : kNarrowRowsSlim;
}
// The affine formats have no wide kernels: their projections own columns from here on (4-bit, 12288 x 2048, us, split /
// owned: 300 rows 37 / 37, 400 rows 50 / 52, 512 rows 56 / 51, 600 rows 68 / 61, 2000 rows 207 / 187).
constexpr int kTallFromAffine = 448;
// Pairs an expert below which the routed experts take them: above that an expert is three tiles of 64 and more, and one unpacking for
// all its rows pays. Prompts through 256 experts of 8 a token, ms, here / there: 1600 tokens 21.7 / 24.4, 2000 24.8 / 27.0, 2400 28.2 / 29.8, 2600
// 31.6 / 31.4, 3000 35.3 / 34.3, 4096 44.7 / 42.2 (80 is 2560 tokens).
constexpr int kNarrowPairs = 80;

// an expert-sorted pair list in device memory, tiles of up to `rows` pairs
struct Plan {
  uint32_t *pair, *tile_expert, *tile_start, *tile_count, *n_tiles;
  uint32_t* expert_at;  // [E] where an expert's pairs begin
  size_t tiles_max;
  int rows;
};

// up to four matrices of one K over the same activations
bool plain_ok(const ornith_linear* const* ws, int n, const void* d_x, int M, void* const* d_ys);
// ... with up to two dense bf16 matrices over the same rows beside them (riders_ok: K and the size too)
bool riders_ok(ornith_ctx* ctx, const ornith_linear* const* ws, int n, int K, int M);
int plain(ornith_ctx* ctx, const ornith_linear* const* ws, int n, const void* d_x, int M, void* const* d_ys,
          const ornith_linear* const* riders = nullptr, int n_riders = 0, void* const* d_yr = nullptr);
// rows of a plan tile
int tile_rows(int pairs, int E);
bool experts_ok(const ornith_kmatrix* w, const void* d_x, size_t x_rows, const void* d_y);
// y[p] = x[row of pair p] . w[expert of p]; with `shared`, pairs + t is token t through that matrix
int gathered(ornith_ctx* ctx, const ornith_kmatrix* w, const ornith_linear* shared, const void* d_x, int pairs, int up_div,
             const Plan& p, void* d_y);
// act[p] = swiglu of the gate and up rows, routed and shared
int gate_up(ornith_ctx* ctx, const ornith_moe_weights* w, const void* d_x, int pairs, const Plan& p, void* d_act);
bool moe_ok(const ornith_moe_weights* w, const void* d_x, int T, const void* d_act, const void* d_y);

// the launches of a family; the first one on a context's device raises the kernels' LDS limits
int launch_kq(ornith_ctx* ctx, const Args& a, int mode, int ct, int rows, int kind, dim3 grid, int lds);
int launch_affine(ornith_ctx* ctx, const Args& a, int mode, int ct, int rows, int kind, dim3 grid, int lds);

}  // namespace nmm

// The kernels of a family, gathered ones for launches of one kind (K1, K2) and of both (-1): a kernel has the registers of
// its widest path. A workgroup is four wavefronts, one a SIMD; a compute unit holds two plain ones, and as many
// gathered ones as registers and LDS allow (WAVES: asked for, a SIMD). TALL1, TALL2: the kernels of kTall, if the family has them.
#define NMM_KERNELS(NAME, AFF, K1, K2, WAVES, LDS_BIT, TALL1, TALL2)                                                \
  template <int CT, int ROWS>                                                                                       \
  __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void NAME##_plain_kernel(Args a) {   \
    body<AFF, CT, kPlain, ROWS, 4>(a);                                                                              \
  }                                                                                                                 \
  template <int MODE, int ROWS, int KIND>                                                                           \
  __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WAVES(KIND, ROWS)))) void                    \
      NAME##_gather_kernel(Args a) {                                                                                \
    body<AFF, 2, MODE, ROWS, 4, KIND>(a);                                                                           \
  }                                                                                                                 \
  int launch_##NAME(ornith_ctx* ctx, const Args& a, int mode, int ct, int rows, int kind, dim3 grid, int lds) {     \
    typedef void (*Kernel)(Args);                                                                                   \
    static const Kernel plain[3][2] = {{NAME##_plain_kernel<1, 32>, NAME##_plain_kernel<1, 64>},                    \
                                       {NAME##_plain_kernel<2, 32>, NAME##_plain_kernel<2, 64>},                    \
                                       {NAME##_plain_kernel<4, 64>, NAME##_plain_kernel<4, 64>}};                   \
    static const Kernel tall[2] = {TALL1, TALL2};                                                                   \
    static const Kernel gather[3][2][3] = {                                                                         \
        {{NAME##_gather_kernel<kGather, 16, K1>, NAME##_gather_kernel<kGather, 32, K1>, NAME##_gather_kernel<kGather, 64, K1>},     \
         {NAME##_gather_kernel<kGateUp, 16, K1>, NAME##_gather_kernel<kGateUp, 32, K1>, NAME##_gather_kernel<kGateUp, 64, K1>}},    \
        {{NAME##_gather_kernel<kGather, 16, K2>, NAME##_gather_kernel<kGather, 32, K2>, NAME##_gather_kernel<kGather, 64, K2>},     \
         {NAME##_gather_kernel<kGateUp, 16, K2>, NAME##_gather_kernel<kGateUp, 32, K2>, NAME##_gather_kernel<kGateUp, 64, K2>}},    \
        {{NAME##_gather_kernel<kGather, 16, -1>, NAME##_gather_kernel<kGather, 32, -1>, NAME##_gather_kernel<kGather, 64, -1>},     \
         {NAME##_gather_kernel<kGateUp, 16, -1>, NAME##_gather_kernel<kGateUp, 32, -1>, NAME##_gather_kernel<kGateUp, 64, -1>}}};   \
    if (!(ctx->lds_attr_set & LDS_BIT)) {                                                                           \
      for (const auto& p : plain)                                                                                   \
        for (const Kernel k : p)                                                                                    \
          ORN_HIP(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes));      \
      for (const Kernel k : tall)                                                                                   \
        if (k) ORN_HIP(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes));        \
      for (const auto& g : gather)                                                                                  \
        for (const auto& m : g)                                                                                     \
          for (const Kernel k : m)                                                                                  \
            ORN_HIP(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes));    \
      ctx->lds_attr_set |= LDS_BIT;                                                                                 \
    }                                                                                                               \
    const int of = kind == K1 ? 0 : kind == K2 ? 1 : 2;                                                             \
    const Kernel k = mode == kPlain ? plain[ct / 2][rows / 64] : mode == kTall ? tall[of != 0] : gather[of][mode == kGateUp][rows / 32]; \
    hipLaunchKernelGGL(k, grid, dim3(256), lds, ctx->stream, a);                                                    \
    ORN_LAUNCH_CHECK("nmm::" #NAME);                                                                                \
    return ORNITH_OK;                                                                                               \
  }
