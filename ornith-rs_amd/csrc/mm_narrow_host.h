// Host side of the few-row GEMM: what the dispatches of linear.hip, kq_mm.hip and moe.hip ask and
// call, and the kernels of one weight family.
#pragma once

#include "mm_narrow.h"

namespace nmm {

// Rows up to which a k-quant projection takes these kernels: the wide kernels' 256 x 128 tiles fill the device from about a
// thousand rows of 12288 columns on, and for up to 2048 columns not before a thousand rows either (2048 x 4096, us here /
// there: 64 rows 7.2 / 52, 256 rows 15 / 53, 700 rows 29 / 54, 1024 rows 38 / 55; 256 x 2048: 5 / 29, 1024 rows 9 / 29).
// More columns than that go to the own-column kernel of kq_mm_own.hip (12288 x 2048 Q4_K, us, here / there: 128 rows 20 / 25, 200 rows
// 27 / 26; the rule there looks at one matrix at a time, never at what shares its launch: a matrix gives the same bits alone and in company).
// The lines for up to 2048 columns, from K = 2048 on (below, the wide kernels' few slabs are over as soon: 2048 x 512 at 1024 rows 10.5 /
// 9.9): Q4_K 1536 rows (2048 x 4096 at 1200 / 1500 / 2000 rows 44 / 54, 46 / 55, 58 / 57), Q6_K 1024 (2048 x 4096 at 1024 / 1200 / 1500 rows
// 51 / 57, 56 / 57, 67 / 58), and up to 256 columns, which are 16 to 40 workgroups of the wide kernels, 2560 (the router at 1200 / 2000 / 2500
// rows 13 / 29, 17 / 29, 21 / 29; level at 4096).
constexpr int kNarrowRows = 192, kNarrowRowsSlim = 1024, kNarrowRowsSlimQ4K = 1536, kNarrowRowsSlimmest = 2560;
// The affine formats have no wide kernels: their projections own columns from here on (4-bit, 12288 x 2048, us, split /
// owned: 300 rows 37 / 37, 400 rows 50 / 52, 512 rows 56 / 51, 600 rows 68 / 61, 2000 rows 207 / 187).
constexpr int kTallFromAffine = 448;
// Pairs an expert below which the routed experts take them: above that an expert is three tiles of 64 and more, and the wide kernels'
// one unpacking for all its rows pays. Prompts through 256 experts of 8 a token, ms, here / there: 1600 tokens 24.9 / 26.8, 2000
// 28.4 / 29.5, 2400 31.4 / 32.6, 2700 35.0 / 35.6, 3000 37.2 / 37.4, 3500 42.0 / 42.1, 4096 47.3 / 46.5, 5000 59.2 / 57.7 (80 is 2560 tokens: past
// that the two are level).
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
