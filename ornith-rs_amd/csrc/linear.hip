// The non-k-quant projections and the polymorphic Linear.
//
// Replaces Linear::matmul (/root/reference/src/ops/linear.rs:23-110), the 8-bit
// affine mat-vec `affine_qmv_fast` (/root/reference/src/ops/quantized.rs:311-333,
// vendored quantized.h:283-289,756-821), the dense bf16 mat-vec and its gathered
// form (/root/reference/src/ops/matmul.rs:334-438,649-) and the embedding lookup
// (/root/reference/src/ops/embedding.rs:18-46).
//
// The mat-vecs here are one wavefront per output row: lane l owns the 8-element (4-bit codes: 16-element)
// chunks j = l + 64c in ascending c, accumulates them in fp32 and the 64 lane sums go through the
// butterfly. Affine matrices of 1024, 2048 and 4096 columns take the kernels of affine_mv.hip instead, with
// the same sums (the row-a-wavefront ones read every weight once an activation row and in one trip to memory
// a chunk: 12288 x 2048 in 4 bits at two rows 15.9 us here with the norm in front, 9.7 there), and prompts
// of ornith_option_gemm_rows() rows and more the matrix cores (mm_narrow.h, kq_mm.hip, dense_mm_kernel below).
#include "dmath.h"
#include "kq_mm_own.h"
#include "linear_device.h"
#include "mm_narrow_host.h"
#include "norm_device.h"
#include "rt.h"

// kquant.hip
extern "C" int kq_qmv_multi_prenorm(ornith_ctx* ctx, const ornith_kmatrix* const* ws, int n,
                                    const void* d_res, const void* d_y, const void* d_wnorm, float eps,
                                    int M, void* d_h_out, void* d_normed_out, void* const* d_ys);

// affine_mv.hip
int affine_mv_multi(ornith_ctx* ctx, const ornith_linear* const* ws, int n, const void* d_x, int M, void* const* d_ys,
                    const PreNorm* pre);

namespace {

// ---- 8-bit affine, group 64 ---------------------------------------------
__global__ __launch_bounds__(64) void affine8_qmv_kernel(const uint8_t* w, const bf16_t* scales,
                                                         const bf16_t* biases, const bf16_t* x,
                                                         bf16_t* y, int O, int K) {
  const int o = blockIdx.x, m = blockIdx.y, lane = threadIdx.x;
  const uint8_t* wr = w + (size_t)o * K;
  const bf16_t* sr = scales + (size_t)o * (K / 64);
  const bf16_t* br = biases + (size_t)o * (K / 64);
  const bf16_t* xr = x + (size_t)m * K;
  const float v = affine8_row_dot(wr, sr, br, xr, K, lane);
  if (lane == 0) y[(size_t)m * O + o] = dm_f2bf(v);
}

// ---- 4-bit affine, group 32 ------------------------------------------------
// One wavefront per output row (four rows a workgroup); lane l owns the 16-element chunks
// j = l + 64c: 8 code bytes and 16 activations, both one aligned load. GATHER selects the
// expert and the activation row through lhs / rhs.
template <bool GATHER>
__global__ __launch_bounds__(256) void affine4_qmv_kernel(const uint8_t* w, const bf16_t* scales,
                                                          const bf16_t* biases, const bf16_t* x, bf16_t* y,
                                                          int E, int O, int K, int x_rows, const uint32_t* lhs,
                                                          const uint32_t* rhs) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int o = blockIdx.x * 4 + wave, r = blockIdx.y;
  if (o >= O) return;
  size_t row = o, xi = r;
  if constexpr (GATHER) {
    xi = min(lhs[r], (uint32_t)(x_rows - 1));
    row = (size_t)min(rhs[r], (uint32_t)(E - 1)) * O + o;
  }
  const uint8_t* wr = w + row * (K / 2);
  const bf16_t* sr = scales + row * (K / 32);
  const bf16_t* br = biases + row * (K / 32);
  const bf16_t* xr = x + xi * K;
  const float v = affine4_row_dot(wr, sr, br, xr, K, lane);
  if (lane == 0) y[(size_t)r * O + o] = dm_f2bf(v);
}

// ---- dense bf16 ------------------------------------------------------------
// grid.x covers rows four at a time (one per wavefront), grid.y is the
// activation row; GATHER selects expert / activation row through lhs, rhs.
// Up to four matrices over the same activations in one launch: the rows of the
// segments follow each other along grid.x, each segment with its own output.
struct DenseSegs {
  const bf16_t* w[4];
  bf16_t* y[4];
  int O[4];
  int n;
};

template <bool GATHER>
__global__ __launch_bounds__(256) void dense_gemv_kernel(DenseSegs s, const bf16_t* x, int K, int E,
                                                         int x_rows, const uint32_t* lhs,
                                                         const uint32_t* rhs) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int o = blockIdx.x * 4 + wave;
  const bf16_t* w = s.w[0];
  bf16_t* y = s.y[0];
  int O = s.O[0];
#pragma unroll
  for (int i = 1; i < 4; ++i) {
    if (i < s.n && o >= O) {
      o -= O;
      w = s.w[i];
      y = s.y[i];
      O = s.O[i];
    }
  }
  if (o >= O) return;
  const int r = blockIdx.y;
  const bf16_t* wr;
  const bf16_t* xr;
  if constexpr (GATHER) {
    const uint32_t xi = min(lhs[r], (uint32_t)(x_rows - 1));
    const uint32_t ei = min(rhs[r], (uint32_t)(E - 1));
    wr = w + ((size_t)ei * O + o) * K;
    xr = x + (size_t)xi * K;
  } else {
    wr = w + (size_t)o * K;
    xr = x + (size_t)r * K;
  }
  const float v = dense_row_dot(wr, xr, K, lane);
  if (lane == 0) y[(size_t)r * O + o] = dm_f2bf(v);
}

// ---- embedding: out = bf16(bf16(q * scale) + bias) ------------------------------
__global__ void embedding_kernel(const uint8_t* w, const bf16_t* scales, const bf16_t* biases,
                                 const uint32_t* ids, bf16_t* out, int V, int K) {
  const int r = blockIdx.y;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= K) return;
  const size_t row = min(ids[r], (uint32_t)(V - 1));
  const float s = dm_bf2f(scales[row * (K / 64) + i / 64]);
  const float b = dm_bf2f(biases[row * (K / 64) + i / 64]);
  const float v = dm_rb((float)w[row * K + i] * s);
  out[(size_t)r * K + i] = dm_f2bf(v + b);
}

// 4-bit table rows: out = bf16(bf16(q * scale) + bias)
__global__ void embedding4_kernel(const uint8_t* w, const bf16_t* scales, const bf16_t* biases,
                                  const uint32_t* ids, bf16_t* out, int V, int K) {
  const int r = blockIdx.y;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= K) return;
  const size_t row = min(ids[r], (uint32_t)(V - 1));
  const uint8_t byte = w[row * (K / 2) + i / 2];
  const float q = (float)((i & 1) ? (byte >> 4) : (byte & 0xF));
  const float s = dm_bf2f(scales[row * (K / 32) + i / 32]);
  const float b = dm_bf2f(biases[row * (K / 32) + i / 32]);
  out[(size_t)r * K + i] = dm_f2bf(dm_rb(q * s) + b);
}

// ---- dense bf16 at prefill widths: a small GEMM on the matrix cores -------------------
// y[M, O] = x[M, K] . W[O, K]^T for the narrow dense projections (the gated-delta a / b heads,
// the shared expert's gate: O of 1 .. 64): as mat-vecs every activation row is read by O / 4
// workgroups. One workgroup = 16 rows; its wavefronts split K and add up through LDS; a
// wavefront feeds v_mfma_f32_16x16x32_bf16 straight from global memory (A: 16 rows x 32
// channels, B: 16 outputs x 32 channels, 16 bytes a lane each). grid.y covers O in NT tiles of 16.
// A launch is one latency chain of some workgroups, so K goes over as many wavefronts as it
// divides into 128-channel pieces (up to 16) and a wavefront asks for a piece's operands at once: 2 x 32
// outputs of K = 2048, 51 / 700 / 6621 rows, with four wavefronts 24.4 / 24.5 / 25.5 us, with sixteen (four tiles)
// 11.6 / 11.8 / 22.0. What bounds it is the L1: sixteen lanes in a row ask for sixteen lines, 64 clocks a load, 320 loads a
// workgroup with four tiles. One tile a workgroup asks 128 times: 5.9 / 6.0 us.
typedef __bf16 dmm_bf16x8_t __attribute__((ext_vector_type(8)));
typedef float dmm_f32x4_t __attribute__((ext_vector_type(4)));

struct DenseMmSegs {
  const bf16_t* w[4];
  bf16_t* y[4];
  int O[4];
  int n;
};

template <int NW, int NT>
__global__ __launch_bounds__(64 * NW) void dense_mm_kernel(DenseMmSegs s, const bf16_t* x, int M, int K) {
  __shared__ __attribute__((aligned(16))) dmm_f32x4_t red[NW][NT][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, lg = lane >> 4;
  const int row0 = blockIdx.x * 16;
  const int kw = K / NW, k0 = wave * kw;  // a multiple of 32
  const bf16_t* xp = x + (size_t)min(row0 + l16, M - 1) * K + k0 + 8 * lg;
  // the 16-output tiles of this workgroup: tile NT * blockIdx.y + nt of the segments' tiles laid end to end (a
  // segment's last tile may be ragged)
  const bf16_t* wp[NT];
  bf16_t* yp[NT];
  int ocol[NT], oend[NT], ostride[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    int t = NT * blockIdx.y + nt, seg = -1;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (seg < 0 && i < s.n) {
        const int tiles = (s.O[i] + 15) / 16;
        if (t < tiles) seg = i; else t -= tiles;
      }
    const int sg = seg < 0 ? 0 : seg;
    ocol[nt] = 16 * t + l16;
    oend[nt] = seg < 0 ? 0 : s.O[sg];
    ostride[nt] = s.O[sg];
    yp[nt] = s.y[sg];
    wp[nt] = s.w[sg] + (size_t)min(ocol[nt], s.O[sg] - 1) * K + k0 + 8 * lg;
  }
  dmm_f32x4_t acc[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) acc[nt] = dmm_f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int k = 0; k < kw; k += 32) {
    const dmm_bf16x8_t a = *reinterpret_cast<const dmm_bf16x8_t*>(xp + k);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
      if (NT == 1 || oend[nt] > 0) {  // (the same for every lane of the wavefront; a single tile is always one of the launch's)
        const dmm_bf16x8_t b = *reinterpret_cast<const dmm_bf16x8_t*>(wp[nt] + k);
        acc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[nt], 0, 0, 0);
      }
  }
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) red[wave][nt][lane] = acc[nt];
  __syncthreads();
  if (wave >= NT) return;
  // output tile nt = wave: D[m = 4 * lg + r][n = l16]
  dmm_f32x4_t v = red[0][wave][lane];
#pragma unroll
  for (int w = 1; w < NW; ++w) v += red[w][wave][lane];
  int col = 0, end = 0, stride = 0;
  bf16_t* y = nullptr;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
    if (nt == wave) {
      col = ocol[nt];
      end = oend[nt];
      stride = ostride[nt];
      y = yp[nt];
    }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = row0 + 4 * lg + r;
    if (col < end && row < M) y[(size_t)row * stride + col] = dm_f2bf(v[r]);
  }
}

// up to four dense matrices of one K over the same activations at prefill width; false when
// the shapes do not allow it
static bool launch_dense_mm(ornith_ctx* ctx, const ornith_linear* const* ws, int n, const void* d_x, int M,
                            void* const* d_ys) {
  if (n < 1 || n > 4 || ((uintptr_t)d_x & 15) != 0) return false;
  DenseMmSegs s{};
  s.n = n;
  int tiles = 0;
  for (int i = 0; i < n; ++i) {
    if (ws[i]->mode != ORNITH_LIN_DENSE || !ws[i]->d_w || ws[i]->K != ws[0]->K || ws[i]->K % 128 != 0 || ws[i]->O < 1 ||
        ((uintptr_t)ws[i]->d_w & 15) != 0)
      return false;
    s.w[i] = (const bf16_t*)ws[i]->d_w;
    s.y[i] = (bf16_t*)d_ys[i];
    s.O[i] = ws[i]->O;
    tiles += (ws[i]->O + 15) / 16;
  }
  // One tile a workgroup while two workgroups a compute unit hold them all (a single tile always:
  // 5.2 -> 4.9 us, at 6621 rows 8.8 -> 6.9); past that the rows read four times cost more than the loads' time divided by four
  // saves. Four tiles, us, four a workgroup / one: 51 rows 11.6 / 5.9, 700 11.8 / 6.0, 1500 11.9 / 9.7, 2048 (two a unit) 11.9 / 9.5, 3000
  // 12.0 / 12.9, 6621 22.0 / 28.5.
  const int rt = (M + 15) / 16, K = ws[0]->K;
  const bool one = tiles == 1 || (long)rt * tiles <= 2L * ctx->compute_units;
  const dim3 grid(rt, one ? tiles : (tiles + 3) / 4);
  typedef void (*Kernel)(DenseMmSegs, const bf16_t*, int, int);
  static const Kernel kernels[3][2] = {{dense_mm_kernel<16, 4>, dense_mm_kernel<16, 1>},
                                       {dense_mm_kernel<8, 4>, dense_mm_kernel<8, 1>},
                                       {dense_mm_kernel<4, 4>, dense_mm_kernel<4, 1>}};
  const int form = K % 2048 == 0 ? 0 : K % 1024 == 0 ? 1 : 2;
  hipLaunchKernelGGL(kernels[form][one], grid, dim3(1024 >> form), 0, ctx->stream, s, (const bf16_t*)d_x, M, K);
  return true;
}

template <bool GATHER>
int launch_dense(ornith_ctx* ctx, const DenseSegs& s, const void* d_x, int K, int E, int x_rows,
                 const uint32_t* d_lhs, const uint32_t* d_rhs, int rows) {
  int total = 0;
  for (int i = 0; i < s.n; ++i) total += s.O[i];
  hipLaunchKernelGGL(dense_gemv_kernel<GATHER>, dim3((total + 3) / 4, rows), dim3(256), 0, ctx->stream, s,
                     (const bf16_t*)d_x, K, E, x_rows, d_lhs, d_rhs);
  ORN_LAUNCH_CHECK(GATHER ? "dense_gemv_kernel<gather>" : "dense_gemv_kernel");
  return ORNITH_OK;
}

}  // namespace

// Several stacked expert tensors [E, O, K] gathered over the same (activation row, expert)
// pairs in one launch (the gate and up projections of dense experts).
extern "C" int dense_gather_mv_multi(ornith_ctx* ctx, const void* const* d_ws, int n, int E, int O, int K,
                                     const void* d_x, int x_rows, const uint32_t* d_lhs,
                                     const uint32_t* d_rhs, int rows, void* const* d_ys) {
  ORN_REQUIRE(ctx && d_ws && d_ys && d_x && d_lhs && d_rhs && n >= 1 && n <= 4, "dense_gather_mv_multi: bad argument");
  ORN_REQUIRE(E >= 1 && O >= 1 && K % 8 == 0 && x_rows >= 1 && rows >= 0 && rows <= 65535,
              "dense_gather_mv: E=%d O=%d K=%d rows=%d", E, O, K, rows);
  if (rows == 0) return ORNITH_OK;
  DenseSegs s{};
  s.n = n;
  for (int i = 0; i < n; ++i) {
    ORN_REQUIRE(d_ws[i] && d_ys[i], "dense_gather_mv_multi: null entry %d", i);
    s.w[i] = (const bf16_t*)d_ws[i];
    s.y[i] = (bf16_t*)d_ys[i];
    s.O[i] = O;
  }
  return launch_dense<true>(ctx, s, d_x, K, E, x_rows, d_lhs, d_rhs, rows);
}

// `wide`: prompt widths, matrix-core GEMMs where the shapes allow; otherwise every row as if alone.
static int linear_matmul(ornith_ctx* ctx, const ornith_linear* w, const void* d_x, int M, void* d_y, bool wide) {
  ORN_REQUIRE(ctx && w && d_x && d_y, "linear_matmul: null argument");
  ORN_REQUIRE(M >= 1, "linear_matmul: M=%d", M);
  switch (w->mode) {
    case ORNITH_LIN_KQUANT:
      ORN_REQUIRE(w->km.O == w->O && w->km.K == w->K, "linear_matmul: k-quant dims disagree");
      // kquant::matmul (src/ops/kquant.rs:783-800): rows within the exact window go through
      // the mat-vec (each row as if alone), prefill widths through the matrix cores
      if (wide && nmm::plain_ok(&w, 1, d_x, M, &d_y)) return nmm::plain(ctx, &w, 1, d_x, M, &d_y);
      if (wide) return ornith_kq_matmul(ctx, &w->km, d_x, M, d_y);
      return ornith_kq_qmv(ctx, &w->km, d_x, ORNITH_BF16, M, d_y, ORNITH_BF16);
    case ORNITH_LIN_AFFINE8:
      ORN_REQUIRE(w->d_w && w->d_scales && w->d_biases, "linear_matmul: affine tensor missing");
      ORN_REQUIRE(w->K % 64 == 0 && w->O >= 1 && M <= 65535, "linear_matmul: affine O=%d K=%d",
                  w->O, w->K);
      if (wide && nmm::plain_ok(&w, 1, d_x, M, &d_y)) return nmm::plain(ctx, &w, 1, d_x, M, &d_y);
      if (const int rc = affine_mv_multi(ctx, &w, 1, d_x, M, &d_y, nullptr); rc >= 0) return rc;
      hipLaunchKernelGGL(affine8_qmv_kernel, dim3(w->O, M), dim3(64), 0, ctx->stream,
                         (const uint8_t*)w->d_w, (const bf16_t*)w->d_scales,
                         (const bf16_t*)w->d_biases, (const bf16_t*)d_x, (bf16_t*)d_y, w->O, w->K);
      ORN_LAUNCH_CHECK("affine8_qmv_kernel");
      return ORNITH_OK;
    case ORNITH_LIN_AFFINE4:
      ORN_REQUIRE(w->d_w && w->d_scales && w->d_biases, "linear_matmul: affine tensor missing");
      ORN_REQUIRE(w->K % 32 == 0 && w->O >= 1 && M <= 65535, "linear_matmul: 4-bit affine O=%d K=%d", w->O, w->K);
      if (wide && nmm::plain_ok(&w, 1, d_x, M, &d_y)) return nmm::plain(ctx, &w, 1, d_x, M, &d_y);
      if (const int rc = affine_mv_multi(ctx, &w, 1, d_x, M, &d_y, nullptr); rc >= 0) return rc;
      hipLaunchKernelGGL(affine4_qmv_kernel<false>, dim3((w->O + 3) / 4, M), dim3(256), 0, ctx->stream,
                         (const uint8_t*)w->d_w, (const bf16_t*)w->d_scales, (const bf16_t*)w->d_biases,
                         (const bf16_t*)d_x, (bf16_t*)d_y, 1, w->O, w->K, M, (const uint32_t*)nullptr,
                         (const uint32_t*)nullptr);
      ORN_LAUNCH_CHECK("affine4_qmv_kernel");
      return ORNITH_OK;
    case ORNITH_LIN_DENSE:
      ORN_REQUIRE(w->d_w, "linear_matmul: dense weight missing");
      ORN_REQUIRE(w->K % 8 == 0 && w->O >= 1 && M <= 65535, "linear_matmul: dense O=%d K=%d", w->O,
                  w->K);
      // prefill widths (outside the exact window, like the k-quant GEMM): on the matrix cores
      if (wide && launch_dense_mm(ctx, &w, 1, d_x, M, &d_y)) {
        ORN_LAUNCH_CHECK("dense_mm_kernel");
        return ORNITH_OK;
      }
      {
        DenseSegs s{};
        s.n = 1;
        s.w[0] = (const bf16_t*)w->d_w;
        s.y[0] = (bf16_t*)d_y;
        s.O[0] = w->O;
        return launch_dense<false>(ctx, s, d_x, w->K, 1, M, nullptr, nullptr, M);
      }
    default:
      return ornith_fail(ORNITH_ERR_INVALID, "linear_matmul: unknown mode %d", w->mode);
  }
}

static int linear_matmul_multi(ornith_ctx* ctx, const ornith_linear* const* ws, int n, const void* d_x, int M,
                               void* const* d_ys, bool wide) {
  ORN_REQUIRE(ctx && ws && d_x && d_ys && n >= 1, "linear_matmul_multi: bad argument");
  bool fuse = ornith_option_fuse_proj() && n >= 2 && n <= 4 && !wide;
  for (int i = 0; i < n; ++i) {
    ORN_REQUIRE(ws[i] && d_ys[i], "linear_matmul_multi: null entry %d", i);
    fuse = fuse && ws[i]->mode == ws[0]->mode && ws[i]->K == ws[0]->K;
    if (ws[i]->mode == ORNITH_LIN_KQUANT) fuse = fuse && ws[i]->km.kind == ws[0]->km.kind;
  }
  // affine matrices share a launch whatever their width in bits
  if (ornith_option_fuse_proj() && n >= 2 && !wide)
    if (const int rc = affine_mv_multi(ctx, ws, n, d_x, M, d_ys, nullptr); rc >= 0) return rc;
  if (fuse && ws[0]->mode == ORNITH_LIN_KQUANT) {
    const ornith_kmatrix* kms[4];
    for (int i = 0; i < n; ++i) kms[i] = &ws[i]->km;
    return ornith_kq_qmv_multi(ctx, kms, n, d_x, ORNITH_BF16, M, d_ys, ORNITH_BF16);
  }
  if (fuse && ws[0]->mode == ORNITH_LIN_DENSE && ws[0]->K % 8 == 0 && M <= 65535) {
    DenseSegs s{};
    s.n = n;
    for (int i = 0; i < n; ++i) {
      ORN_REQUIRE(ws[i]->d_w && ws[i]->O >= 1, "linear_matmul_multi: dense weight %d missing", i);
      s.w[i] = (const bf16_t*)ws[i]->d_w;
      s.y[i] = (bf16_t*)d_ys[i];
      s.O[i] = ws[i]->O;
    }
    return launch_dense<false>(ctx, s, d_x, ws[0]->K, 1, M, nullptr, nullptr, M);
  }
  // Prefill widths: the matrices that take the few-row GEMM share a launch of it (all of them, or the
  // ones with few columns of a wider call), narrow dense ones ride along; the others go on below, the dense ones among themselves.
  if (wide && ornith_option_fuse_proj() && n >= 2 && n <= 4) {
    const ornith_linear *few[4], *dense[4], *rest[4];
    void *yf[4], *yd[4], *yr[4];
    int nf = 0, nd = 0, nr = 0;
    for (int i = 0; i < n; ++i) {
      const bool ok = nmm::plain_ok(&ws[i], 1, d_x, M, &d_ys[i]), plain_dense = ws[i]->mode == ORNITH_LIN_DENSE;
      (ok ? few[nf] : plain_dense ? dense[nd] : rest[nr]) = ws[i];
      (ok ? yf[nf++] : plain_dense ? yd[nd++] : yr[nr++]) = d_ys[i];
    }
    // (a single one, too: in a launch of the wide kernels it would have other sums than alone)
    const bool shared = nf >= 1 && nmm::plain_ok(few, nf, d_x, M, yf);
    if (shared || (nd && nd < n)) {
      const bool riding = shared && nmm::riders_ok(ctx, dense, nd, few[0]->K, M);
      int rc = ORNITH_OK;
      if (shared) rc = nmm::plain(ctx, few, nf, d_x, M, yf, dense, riding ? nd : 0, yd);
      else
        for (int i = 0; i < nf; ++i) {
          rest[nr] = few[i];
          yr[nr++] = yf[i];
        }
      if (!rc && nr) rc = linear_matmul_multi(ctx, rest, nr, d_x, M, yr, wide);
      if (!rc && nd && !riding) rc = linear_matmul_multi(ctx, dense, nd, d_x, M, yd, wide);
      return rc;
    }
  }
  // ... dense matrices of one K likewise
  if (wide && ornith_option_fuse_proj() && n >= 2 && launch_dense_mm(ctx, ws, n, d_x, M, d_ys)) {
    ORN_LAUNCH_CHECK("dense_mm_kernel");
    return ORNITH_OK;
  }
  // prefill widths: runs of k-quant matrices of one K share a GEMM launch. Those that suit the own-column form may always; of
  // others a run of one kind may be large (it picks its tile by size), but a matrix of the other kind joins a run only
  // while the run is narrow (a mixed launch takes 128-row tiles, which wide matrices should not pay for).
  for (int i = 0; i < n;) {
    int j = i + 1;
    if (wide && ornith_option_fuse_proj() && ws[i]->mode == ORNITH_LIN_KQUANT) {
      int cols = ws[i]->O;
      bool mixed = false, own = kq_mm_own_suits(ws[i]->km, d_x, M);
      while (j < n && j - i < 4 && ws[j]->mode == ORNITH_LIN_KQUANT && ws[j]->K == ws[i]->K) {
        const bool other = ws[j]->km.kind != ws[i]->km.kind;
        own = own && kq_mm_own_suits(ws[j]->km, d_x, M);
        if ((other || mixed) && !own && cols + ws[j]->O > 2048) break;
        mixed = mixed || other;
        cols += ws[j]->O;
        ++j;
      }
    }
    int rc;
    if (j - i >= 2) {
      const ornith_kmatrix* kms[4];
      for (int t = i; t < j; ++t) {
        ORN_REQUIRE(ws[t]->km.O == ws[t]->O && ws[t]->km.K == ws[t]->K, "linear_matmul_multi: k-quant dims disagree");
        kms[t - i] = &ws[t]->km;
      }
      rc = ornith_kq_matmul_multi(ctx, kms, j - i, d_x, M, d_ys + i);
    } else {
      rc = linear_matmul(ctx, ws[i], d_x, M, d_ys[i], wide);
    }
    if (rc) return rc;
    i = j;
  }
  return ORNITH_OK;
}

// The projections of a block whose sums are the exact path's at every width (moe.hip).
int linear_exact_multi(ornith_ctx* ctx, const ornith_linear* const* ws, int n, const void* d_x, int M, void* const* d_ys) {
  return linear_matmul_multi(ctx, ws, n, d_x, M, d_ys, false);
}

extern "C" {

int ornith_linear_matmul(ornith_ctx* ctx, const ornith_linear* w, const void* d_x, int M, void* d_y) {
  return linear_matmul(ctx, w, d_x, M, d_y, M >= kPrefillRows);
}

int ornith_linear_matmul_multi(ornith_ctx* ctx, const ornith_linear* const* ws, int n, const void* d_x, int M,
                               void* const* d_ys) {
  return linear_matmul_multi(ctx, ws, n, d_x, M, d_ys, M >= kPrefillRows);
}

int ornith_add_rms_linear_multi(ornith_ctx* ctx, const ornith_linear* const* ws, int n,
                                const void* d_res, const void* d_y, const void* d_wnorm, float eps, int M,
                                void* d_h_out, void* d_normed_out, void* const* d_ys) {
  ORN_REQUIRE(ctx && ws && d_res && d_y && d_wnorm && d_h_out && d_normed_out && d_ys && n >= 1,
              "add_rms_linear_multi: bad argument");
  for (int i = 0; i < n; ++i) ORN_REQUIRE(ws[i] && d_ys[i], "add_rms_linear_multi: null entry %d", i);
  // the norm in the head of the projections' launch (a call that runs as a GEMM has it in front)
  bool head = ornith_option_fuse_norm() && n <= 4 && M >= 1 && M <= 4 && M < kPrefillRows;
  for (int i = 0; i < n; ++i) head = head && ws[i]->K == kPreN;
  if (head) {
    const PreNorm pre{(const bf16_t*)d_res, (const bf16_t*)d_y, (const bf16_t*)d_wnorm, (bf16_t*)d_h_out, (bf16_t*)d_normed_out, eps};
    head = prenorm_apart(pre, M);
    bool kq = true;
    const ornith_kmatrix* kms[4];
    for (int i = 0; i < n; ++i) {
      head = head && prenorm_apart(pre, M, d_ys[i], (size_t)M * ws[i]->O * 2);
      kq = kq && ws[i]->mode == ORNITH_LIN_KQUANT;
      kms[i] = &ws[i]->km;
    }
    int rc = -1;
    if (head) rc = kq ? kq_qmv_multi_prenorm(ctx, kms, n, d_res, d_y, d_wnorm, eps, M, d_h_out, d_normed_out, d_ys)
                      : affine_mv_multi(ctx, ws, n, nullptr, M, d_ys, &pre);
    if (rc >= 0) return rc;
  }
  int rc = ornith_add_rms_norm(ctx, d_res, d_y, d_wnorm, M, ws[0]->K, eps, d_h_out, d_normed_out);
  if (rc) return rc;
  return ornith_linear_matmul_multi(ctx, ws, n, d_normed_out, M, d_ys);
}

int ornith_dense_gather_mv(ornith_ctx* ctx, const void* d_w, int E, int O, int K, const void* d_x,
                           int x_rows, const uint32_t* d_lhs, const uint32_t* d_rhs, int rows,
                           void* d_y) {
  ORN_REQUIRE(ctx && d_w && d_x && d_lhs && d_rhs && d_y, "dense_gather_mv: null argument");
  ORN_REQUIRE(E >= 1 && O >= 1 && K % 8 == 0 && x_rows >= 1 && rows >= 0 && rows <= 65535,
              "dense_gather_mv: E=%d O=%d K=%d rows=%d", E, O, K, rows);
  if (rows == 0) return ORNITH_OK;
  const void* ws[1] = {d_w};
  void* ys[1] = {d_y};
  return dense_gather_mv_multi(ctx, ws, 1, E, O, K, d_x, x_rows, d_lhs, d_rhs, rows, ys);
}

int ornith_affine4_gather_qmv(ornith_ctx* ctx, const void* d_w, const void* d_scales, const void* d_biases,
                              int E, int O, int K, const void* d_x, int x_rows, const uint32_t* d_lhs,
                              const uint32_t* d_rhs, int rows, void* d_y) {
  ORN_REQUIRE(ctx && d_w && d_scales && d_biases && d_x && d_lhs && d_rhs && d_y, "affine4_gather_qmv: null argument");
  ORN_REQUIRE(E >= 1 && O >= 1 && K % 32 == 0 && x_rows >= 1 && rows >= 0 && rows <= 65535,
              "affine4_gather_qmv: E=%d O=%d K=%d rows=%d", E, O, K, rows);
  if (rows == 0) return ORNITH_OK;
  hipLaunchKernelGGL(affine4_qmv_kernel<true>, dim3((O + 3) / 4, rows), dim3(256), 0, ctx->stream,
                     (const uint8_t*)d_w, (const bf16_t*)d_scales, (const bf16_t*)d_biases, (const bf16_t*)d_x,
                     (bf16_t*)d_y, E, O, K, x_rows, d_lhs, d_rhs);
  ORN_LAUNCH_CHECK("affine4_qmv_kernel<gather>");
  return ORNITH_OK;
}

int ornith_embedding(ornith_ctx* ctx, const ornith_linear* table, const uint32_t* d_ids, int n,
                     void* d_out) {
  ORN_REQUIRE(ctx && table && d_ids && d_out, "embedding: null argument");
  ORN_REQUIRE(table->mode == ORNITH_LIN_AFFINE8 || table->mode == ORNITH_LIN_AFFINE4,
              "embedding: table mode %d; the lookup is defined for the affine tables only",
              table->mode);
  ORN_REQUIRE(table->K % 64 == 0 && n >= 0 && n <= 65535, "embedding: K=%d n=%d", table->K, n);
  if (n == 0) return ORNITH_OK;
  if (table->mode == ORNITH_LIN_AFFINE4) {
    hipLaunchKernelGGL(embedding4_kernel, dim3((table->K + 255) / 256, n), dim3(256), 0, ctx->stream,
                       (const uint8_t*)table->d_w, (const bf16_t*)table->d_scales,
                       (const bf16_t*)table->d_biases, d_ids, (bf16_t*)d_out, table->O, table->K);
    ORN_LAUNCH_CHECK("embedding4_kernel");
    return ORNITH_OK;
  }
  hipLaunchKernelGGL(embedding_kernel, dim3((table->K + 255) / 256, n), dim3(256), 0, ctx->stream,
                     (const uint8_t*)table->d_w, (const bf16_t*)table->d_scales,
                     (const bf16_t*)table->d_biases, d_ids, (bf16_t*)d_out, table->O, table->K);
  ORN_LAUNCH_CHECK("embedding_kernel");
  return ORNITH_OK;
}

}  // extern "C"
