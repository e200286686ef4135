// Element-wise evaluation of the device scalar functions, so a caller can check
// them bit for bit against a CPU evaluation of the same formulae.
#include "dmath.h"
#include "kq_mm_own.h"
#include "mm_narrow_host.h"
#include "rt.h"

namespace {
__global__ void unary_kernel(int op, const float* in, float* out, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float x = in[i];
  float y;
  switch (op) {
    case ORNITH_FN_EXP: y = dm_exp(x); break;
    case ORNITH_FN_LOG: y = dm_log(x); break;
    case ORNITH_FN_LOG1P: y = dm_log1p(x); break;
    case ORNITH_FN_SIGMOID_BF16: {  // and its two-at-a-time form: 2, which is no sigmoid, where they differ
      const float xr = dm_rb(x), n = dm_sigmoid_bf16(-xr);
      float u, v;
      y = dm_sigmoid_bf16(xr);
      dm_sigmoid_bf16x2(xr, -xr, u, v);
      if (y == y && (u != y || v != n)) y = 2.0f;
      break;
    }
    case ORNITH_FN_SIGMOID_F32: y = dm_sigmoid_f32(x); break;
    case ORNITH_FN_RSQRT: y = dm_rsqrt(x); break;
    case ORNITH_FN_RECIP: y = 1.0f / x; break;
    case ORNITH_FN_ROUND_BF16: y = dm_rb(x); break;
    case ORNITH_FN_WAVE_SUM: y = dm_wave_sum<64>(x); break;
    case ORNITH_FN_XOR_LANE + 0: y = dm_xor_lane<1>(x); break;
    case ORNITH_FN_XOR_LANE + 1: y = dm_xor_lane<2>(x); break;
    case ORNITH_FN_XOR_LANE + 2: y = dm_xor_lane<4>(x); break;
    case ORNITH_FN_XOR_LANE + 3: y = dm_xor_lane<8>(x); break;
    case ORNITH_FN_XOR_LANE + 4: y = dm_xor_lane<16>(x); break;
    case ORNITH_FN_XOR_LANE + 5: y = dm_xor_lane<32>(x); break;
    default: y = x;
  }
  out[i] = y;
}
}  // namespace

extern "C" int ornith_selftest_unary(ornith_ctx* ctx, int fn, const float* d_in, float* d_out,
                                     int64_t n) {
  ORN_REQUIRE(ctx && d_in && d_out && n >= 0, "selftest_unary: bad argument");
  ORN_REQUIRE(fn >= 0 && fn <= ORNITH_FN_XOR_LANE + 5, "selftest_unary: unknown function %d", fn);
  // the lane-crossing functions need whole wavefronts: n a multiple of the 256-thread block
  ORN_REQUIRE(fn < ORNITH_FN_WAVE_SUM || n % 256 == 0, "selftest_unary: function %d needs n %% 256 == 0", fn);
  if (n == 0) return ORNITH_OK;
  hipLaunchKernelGGL(unary_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, ctx->stream, fn,
                     d_in, d_out, n);
  ORN_LAUNCH_CHECK("unary_kernel");
  return ORNITH_OK;
}

extern "C" int ornith_selftest_gather_form(const ornith_kmatrix* w, const void* d_x, int pairs, int top_k, int is_up, const void* d_y) {
  if (!w || w->E < 1 || pairs < 1 || top_k < 1) return -1;
  return kq_gather_form(*w, d_x, pairs, top_k, is_up != 0, d_y, 256);
}

extern "C" int ornith_selftest_gemm_form(const ornith_linear* w, const void* d_x, int M, const void* d_y) {
  if (!w || w->mode != ORNITH_LIN_KQUANT) return -1;
  void* const y = const_cast<void*>(d_y);
  if (nmm::plain_ok(&w, 1, d_x, M, &y)) return 3;
  if (!kq_mm_own_suits(w->km, d_x, M)) return 0;
  OwnArgs a{};
  a.m[0].O = w->km.O;
  a.n = 1;
  a.M = M;
  a.K = w->km.K;
  return kq_mm_own_halves(w->km, M) ? 2 : kq_mm_own_thin(a, 256) ? 4 : 1;
}
