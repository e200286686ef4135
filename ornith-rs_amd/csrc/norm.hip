// RMS norms: plain, fused residual add, and the gated output norm of the
// gated-delta layer.
//
// Replaces norm::{rms_norm, add_rms_norm, rms_norm_gated}
// (/root/reference/src/ops/norm.rs:19-220; vendored rms_norm.metal:12-81,
// /root/reference/kernels/ornith_norm.metal:28-183).
//
// Rows up to 512 wide: one wavefront per row (see norm_device.h for the arithmetic and
// its order). Wider rows: one workgroup of n/8 threads per row, eight values (16 bytes)
// per thread, because a single wavefront walking 32 or 64 values per lane through the
// add / round / scale / round steps is a chain of thousands of dependent instructions.
// The element-wise steps are spread over the workgroup; only the sum of squares keeps
// its defined order (lane l of a wavefront owns [l*PER, (l+1)*PER), one fma chain, butterfly), handed from thread to thread.
#include "norm_device.h"
#include "rt.h"

namespace {

template <int PER, int MODE>
__global__ __launch_bounds__(64) void rms_kernel(const bf16_t* a, const bf16_t* b, const bf16_t* w,
                                                 const bf16_t* z, bf16_t* h_out, bf16_t* out, int n,
                                                 float eps) {
  const size_t off = (size_t)blockIdx.x * n;
  rms_row<PER, MODE>(a + off, b ? b + off : nullptr, w, z ? z + off : nullptr,
                     h_out ? h_out + off : nullptr, out + off, n, eps, threadIdx.x);
}

// The gated norm of 128-wide rows (a prompt's value heads: 32 rows a token), sixteen lanes and one 16-byte load a row and operand,
// sixteen rows a workgroup. Bound by the stream (8 bytes a value) behind one trip to memory; a wavefront a row with 4-byte
// loads was a workgroup a row and bound by their launch: us, 51 / 700 / 6621 tokens 4.6 / 7.5 / 55.4 -> 4.4 / 6.8 / 40.9. Lane j holds the values of
// lanes 4 j .. 4 j + 3 of a row's wavefront, whose sum it keeps: strides 32 .. 4 of the butterfly pair lanes, 2 and 1 the four of a lane.
__global__ __launch_bounds__(256) void rms_gated_kernel(const bf16_t* a, const bf16_t* w, const bf16_t* z, bf16_t* out, int rows,
                                                        float eps) {
  constexpr int N = 128;
  const int row = blockIdx.x * 16 + (threadIdx.x >> 4), e0 = 8 * (threadIdx.x & 15);
  const size_t off = (size_t)min(row, rows - 1) * N + e0;
  float x[8], g[8], wv[8], p[4];
  load_bf16<8>(a + off, x);
  load_bf16<8>(z + off, g);
  load_bf16<8>(w + e0, wv);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    p[i] = dm_fma(x[2 * i], x[2 * i], 0.f);
    p[i] = dm_fma(x[2 * i + 1], x[2 * i + 1], p[i]);
    p[i] = p[i] + dm_xor_lane<8>(p[i]);
    p[i] = p[i] + dm_xor_lane<4>(p[i]);
    p[i] = p[i] + dm_xor_lane<2>(p[i]);
    p[i] = p[i] + dm_xor_lane<1>(p[i]);
  }
  const float inv = dm_rsqrt(((p[0] + p[2]) + (p[1] + p[3])) / (float)N + eps);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    x[i] = dm_rb(wv[i] * dm_rb(x[i] * inv));
    x[i] = (g[i] * dm_sigmoid_f32(g[i])) * x[i];
  }
  if (row < rows) store_bf16<8>(out + off, x);
}

template <int PER, int MODE>
__global__ __launch_bounds__(PER * 8) void rms_wide_kernel(const bf16_t* a, const bf16_t* b,
                                                           const bf16_t* w, bf16_t* h_out,
                                                           bf16_t* out, int n, float eps) {
  static_assert(PER % 8 == 0 && MODE != NORM_GATED, "wide rows: plain and add only");
  __shared__ float sums[64];
  const size_t off = (size_t)blockIdx.x * n;
  const int tid = threadIdx.x, e0 = tid * 8;
  float x[8], wv[8];
  load_bf16<8>(a + off + e0, x);
  if (w) load_bf16<8>(w + e0, wv);
  if constexpr (MODE == NORM_ADD) {
    float y[8];
    load_bf16<8>(b + off + e0, y);
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = dm_rb(x[i] + y[i]);
    store_bf16<8>(h_out + off + e0, x);
  }
  const float inv = wide_row_inv<PER>(x, n, eps, sums);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    x[i] = dm_rb(x[i] * inv);
    if (w) x[i] = dm_rb(wv[i] * x[i]);
  }
  store_bf16<8>(out + off + e0, x);
}

template <int MODE>
int launch_rms(ornith_ctx* ctx, const void* a, const void* b, const void* w, const void* z,
               void* h_out, void* out, int rows, int n, float eps, const char* who) {
  ORN_REQUIRE(rows >= 1 && n >= 64 && n % 64 == 0, "%s: rows=%d n=%d", who, rows, n);
  // vector accesses need the row pieces aligned: rows start on n*2 bytes, pieces on PER*2
  const uintptr_t all = (uintptr_t)a | (uintptr_t)b | (uintptr_t)w | (uintptr_t)z | (uintptr_t)h_out |
                        (uintptr_t)out;
  ORN_REQUIRE((all & 15) == 0, "%s: operands must be 16-byte aligned", who);
  if (MODE == NORM_GATED && n == 128) {
    hipLaunchKernelGGL(rms_gated_kernel, dim3((rows + 15) / 16), dim3(256), 0, ctx->stream, (const bf16_t*)a, (const bf16_t*)w,
                       (const bf16_t*)z, (bf16_t*)out, rows, eps);
    ORN_LAUNCH_CHECK("rms_gated_kernel");
    return ORNITH_OK;
  }
#define RMS_CASE(P)                                                                              \
  case P:                                                                                        \
    hipLaunchKernelGGL((rms_kernel<P, MODE>), dim3(rows), dim3(64), 0, ctx->stream,              \
                       (const bf16_t*)a, (const bf16_t*)b, (const bf16_t*)w, (const bf16_t*)z,   \
                       (bf16_t*)h_out, (bf16_t*)out, n, eps);                                    \
    break;
  switch (n / 64) {
    RMS_CASE(1)
    RMS_CASE(2)
    RMS_CASE(4)
    RMS_CASE(8)
#undef RMS_CASE
#define RMS_CASE(P)                                                                              \
  case P:                                                                                        \
    if constexpr (MODE == NORM_GATED)                                                            \
      hipLaunchKernelGGL((rms_kernel<P, MODE>), dim3(rows), dim3(64), 0, ctx->stream,            \
                         (const bf16_t*)a, (const bf16_t*)b, (const bf16_t*)w, (const bf16_t*)z, \
                         (bf16_t*)h_out, (bf16_t*)out, n, eps);                                  \
    else                                                                                         \
      hipLaunchKernelGGL((rms_wide_kernel<P, MODE>), dim3(rows), dim3(P * 8), 0, ctx->stream,    \
                         (const bf16_t*)a, (const bf16_t*)b, (const bf16_t*)w, (bf16_t*)h_out,   \
                         (bf16_t*)out, n, eps);                                                  \
    break;
    RMS_CASE(16)
    RMS_CASE(32)
    RMS_CASE(64)
    default:
      return ornith_fail(ORNITH_ERR_UNSUPPORTED, "%s: row width %d (need 64 * 2^j, j <= 6)", who, n);
  }
#undef RMS_CASE
  ORN_LAUNCH_CHECK("rms_kernel");
  return ORNITH_OK;
}

}  // namespace

extern "C" {

int ornith_rms_norm(ornith_ctx* ctx, const void* d_x, const void* d_w, int rows, int n, float eps,
                    void* d_out) {
  ORN_REQUIRE(ctx && d_x && d_out, "rms_norm: null argument");
  return launch_rms<NORM_PLAIN>(ctx, d_x, nullptr, d_w, nullptr, nullptr, d_out, rows, n, eps,
                                "rms_norm");
}

int ornith_add_rms_norm(ornith_ctx* ctx, const void* d_a, const void* d_b, const void* d_w, int rows,
                        int n, float eps, void* d_h_out, void* d_out) {
  ORN_REQUIRE(ctx && d_a && d_b && d_h_out && d_out, "add_rms_norm: null argument");
  return launch_rms<NORM_ADD>(ctx, d_a, d_b, d_w, nullptr, d_h_out, d_out, rows, n, eps,
                              "add_rms_norm");
}

int ornith_rms_norm_gated(ornith_ctx* ctx, const void* d_y, const void* d_w, const void* d_z,
                          int rows, int n, float eps, void* d_out) {
  ORN_REQUIRE(ctx && d_y && d_w && d_z && d_out, "rms_norm_gated: null argument");
  return launch_rms<NORM_GATED>(ctx, d_y, nullptr, d_w, d_z, nullptr, d_out, rows, n, eps,
                                "rms_norm_gated");
}

}  // extern "C"
