// Q4_K / Q6_K mat-vec of three and more activation rows over large matrices (the output head of a verify
// window, the projections of a short prompt): groups of up
// to four activation rows on the matrix cores, with the fp32 chains of kquant.hip and their order.
//
// v_mfma_f32_4x4x1_16b_f32 is sixteen outer products of four values by four, each product added to
// its element with one rounding: the fused multiply-add of a chain's next step, bit for bit, four
// activation rows by four weight rows by sixteen chunks at once. Lane 4 b + j holds weight row j and
// activation row j of chunk b: it unpacks 1 / 4 of what a lane of the vector form unpacks for the same
// sums, and 256 multiply-adds issue as one instruction of eight clocks where four rows took four
// vector instructions (at two wavefronts a SIMD, which is what 32 activations a row and lane leave
// room for, 9 clocks and more). Lane 4 b + j ends with the sums of weight row j for the four
// activation rows, so scales and minima are applied once per row and chunk as before.
//
// The canonical sum of a row is kept: chunk c's value, chunks c and c + 64 added where a row has 128
// (K = 4096 of Q4_K), then the butterfly over the chunks, strides 32 .. 1. Chunk c = b + 16 s sits in
// lane group b and register set s, so the upper strides pair registers (or the two wavefronts that
// share a row, KS = 2) and the lower ones lanes.
//
// Measured, us, vector form -> this one: 248320 x 2048 of Q4_K at 4 rows 130 -> 111, 26064 x 2048 at 15
// rows 61 -> 47, 30977 x 1024 of Q6_K at 11 rows 36.5 -> 26; level at 12288 x 2048 and 13 rows (24.7 and
// 24.5) and, Q6_K, 9216 x 2048 and 13 rows (22.4 and 23.1), slower below (kq_rows_suits). A third
// wavefront a SIMD, with the activations left packed in bf16, spills: the compiler widens them ahead.
#include <type_traits>

#include "kq_args.h"
#include "kq_device.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int kRows = 4;  // activation rows of a group, weight rows of a wavefront's step

// value of lane (l & ~3) + T of every quad
template <int T>
__device__ __forceinline__ float quad_lane(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), T * 0x55, 0xF, 0xF, true));
}
__device__ __forceinline__ f32x4 quad_all(float v) { return f32x4{quad_lane<0>(v), quad_lane<1>(v), quad_lane<2>(v), quad_lane<3>(v)}; }
__device__ __forceinline__ f32x4 outer(float x, float w, f32x4 acc) { return __builtin_amdgcn_mfma_f32_4x4x1f32(x, w, acc, 0, 0, 0); }

// Byte K of a word as a float for a matrix instruction. Not dm_ubyte: a matrix instruction may not
// follow the vector instruction that made its operand within two wait states, and the compiler, which
// inserts them, does not look into assembly. `opaque` hides the nibble mask from it, with which it would
// take a bit-field extract and a conversion.
__device__ __forceinline__ uint32_t opaque(uint32_t w) {
  asm("" : "+v"(w));
  return w;
}
template <int K>
__device__ __forceinline__ float byte_of(uint32_t w) { return (float)((w >> (8 * K)) & 0xffu); }

// a lane's chunks b + 16 s (+ 16 NS ks) of its activation row, and what they make of a weight row
template <int KIND, int NS>
struct RowsLane;
template <int NS>
struct RowsLane<ORNITH_Q4K, NS> {
  typedef Q4Row Row;
  float xl[NS][16], xh[NS][16];
  f32x4 sl[NS], sh[NS];  // the four activation rows' sums
  int blk0, g, h;        // block of set 0 (set s: two blocks further each), 64-group, half
  __device__ __forceinline__ void place(int b, int ks) {
    blk0 = (b >> 3) + 2 * NS * ks;
    g = (b & 7) >> 1;
    h = b & 1;
  }
  template <bool XF32>
  __device__ __forceinline__ void load_x(const void* xrow) {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int off = 256 * (blk0 + 2 * s) + 64 * g + 16 * h;
      load_x16<XF32>(xrow, off, xl[s]);
      load_x16<XF32>(xrow, off + 32, xh[s]);
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      float a = 0.f, c = 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        a = a + xl[s][i];
        c = c + xh[s][i];
      }
      sl[s] = quad_all(a);
      sh[s] = quad_all(c);
    }
  }
  __device__ __forceinline__ Row load(const KqSeg& sg, int row, int nb, int s) const {
    Row r;
    const int64_t at = (int64_t)row * nb + blk0 + 2 * s;
    r.q = *reinterpret_cast<const uint4*>(sg.qs + at * 128 + 32 * g + 16 * h);
    const uint32_t* sc = reinterpret_cast<const uint32_t*>(sg.scales + at * 12);
    r.s0 = sc[0];
    r.s1 = sc[1];
    r.s2 = sc[2];
    r.dmw = *reinterpret_cast<const uint32_t*>(sg.dm + at * 2);
    return r;
  }
  __device__ __forceinline__ f32x4 chunk(const Row& r, int s) const {
    const uint32_t w[4] = {r.q.x, r.q.y, r.q.z, r.q.w};
    f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = lo;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t wl = opaque(w[k] & 0x0f0f0f0fu), wh = opaque(w[k] & 0xf0f0f0f0u);  // (16 n: see q4_accumulate)
      lo = outer(xl[s][4 * k], byte_of<0>(wl), lo);
      hi = outer(xh[s][4 * k], byte_of<0>(wh), hi);
      lo = outer(xl[s][4 * k + 1], byte_of<1>(wl), lo);
      hi = outer(xh[s][4 * k + 1], byte_of<1>(wh), hi);
      lo = outer(xl[s][4 * k + 2], byte_of<2>(wl), lo);
      hi = outer(xh[s][4 * k + 2], byte_of<2>(wh), hi);
      lo = outer(xl[s][4 * k + 3], byte_of<3>(wl), lo);
      hi = outer(xh[s][4 * k + 3], byte_of<3>(wh), hi);
    }
    const Q4Scales sc(r, g);
    f32x4 p;
#pragma unroll
    for (int t = 0; t < kRows; ++t) p[t] = 0.f + sc.fold(lo[t], hi[t], sl[s][t], sh[s][t]);
    return p;
  }
};
template <int NS>
struct RowsLane<ORNITH_Q6K, NS> {
  typedef Q6Row Row;
  float x[NS][4][16];
  int blk0, n, u;  // set s: four blocks further each; 128-half, half of its positions
  __device__ __forceinline__ void place(int b, int ks) {
    blk0 = (b >> 2) + 4 * NS * ks;
    n = (b & 3) >> 1;
    u = b & 1;
  }
  template <bool XF32>
  __device__ __forceinline__ void load_x(const void* xrow) {
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int g = 0; g < 4; ++g) load_x16<XF32>(xrow, 256 * (blk0 + 4 * s) + 128 * n + 16 * u + 32 * g, x[s][g]);
  }
  __device__ __forceinline__ Row load(const KqSeg& sg, int row, int nb, int s) const {
    Row r;
    const int64_t at = (int64_t)row * nb + blk0 + 4 * s;
    const uint8_t* blk = sg.qs + at * 192;
    r.qa = *reinterpret_cast<const uint4*>(blk + 64 * n + 16 * u);
    r.qb = *reinterpret_cast<const uint4*>(blk + 64 * n + 32 + 16 * u);
    r.qh = *reinterpret_cast<const uint4*>(blk + 128 + 32 * n + 16 * u);
    r.sc = *reinterpret_cast<const uint2*>(sg.scales + at * 16 + 8 * n);
    r.d = sg.dm[at];
    return r;
  }
  __device__ __forceinline__ f32x4 chunk(const Row& r, int s) const {
    f32x4 sum[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) sum[g] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto word = [&](auto kc) {
      constexpr int k = decltype(kc)::value;
      uint32_t c[4];
      q6_codes<k>(r, c);
#pragma unroll
      for (int g = 0; g < 4; ++g) c[g] = opaque(c[g]);
#define ORN_ROWS_STEP(I) \
  _Pragma("unroll") for (int g = 0; g < 4; ++g) sum[g] = outer(x[s][g][4 * k + I], byte_of<I>(c[g]) - 32.0f, sum[g]);
      ORN_ROWS_STEP(0)
      ORN_ROWS_STEP(1)
      ORN_ROWS_STEP(2)
      ORN_ROWS_STEP(3)
#undef ORN_ROWS_STEP
    };
    word(std::integral_constant<int, 0>{});
    word(std::integral_constant<int, 1>{});
    word(std::integral_constant<int, 2>{});
    word(std::integral_constant<int, 3>{});
    const Q6Scales sc(r, u);
    f32x4 p;
#pragma unroll
    for (int t = 0; t < kRows; ++t) p[t] = 0.f + sc.fold(sum[0][t], sum[1][t], sum[2][t], sum[3][t]);
    return p;
  }
};

// grid (row blocks of all segments, groups of activation rows), 256 threads; NS register sets of sixteen
// chunks, KS wavefronts a row
template <int KIND, int NS, int KS, bool XF32>
__global__ __launch_bounds__(256, 2) void kq_rows_kernel(KqArgs a) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, b = lane >> 2, j = lane & 3;
  const int ks = KS == 1 ? 0 : (wave & 1), rw = KS == 1 ? wave : (wave >> 1);
  constexpr int WPB = 4 / KS;
  const int nb = a.K >> 8;
  KqSeg sg = a.seg[0];
#pragma unroll
  for (int i = 1; i < kMaxSeg; ++i)
    if (i < a.nseg && (int)blockIdx.x >= a.seg[i].first_block) sg = a.seg[i];
  const int m0 = blockIdx.y * kRows, O = sg.O;
  const int base = (((int)blockIdx.x - sg.first_block) * WPB + rw) * (kRows * a.iters);
  RowsLane<KIND, NS> L;
  L.place(b, ks);
  typename RowsLane<KIND, NS>::Row row[NS];
  auto fetch = [&](int it, int s) { row[s] = L.load(sg, min(base + kRows * it + j, O - 1), nb, s); };
  __shared__ float part[KS == 2 ? WPB * NS * kRows * 64 : 1];

  // what is small and cached first (loads return in issue order), then the first rows
  L.template load_x<XF32>(static_cast<const char*>(a.x) + (size_t)min(m0 + j, a.x_rows - 1) * a.K * (XF32 ? 4 : 2));
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int s = 0; s < NS; ++s) fetch(0, s);
  for (int it = 0; it < a.iters; ++it) {
    f32x4 p[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      p[s] = L.chunk(row[s], s);
      fetch(min(it + 1, a.iters - 1), s);  // (past the end the last rows again: no load under a condition)
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (KS == 2) {
      float* mine = part + rw * (NS * kRows * 64) + lane;
      __syncthreads();
      if (ks == 1) {
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
          for (int t = 0; t < kRows; ++t) mine[(s * kRows + t) * 64] = p[s][t];
      }
      __syncthreads();
      if (ks == 0) {
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
          for (int t = 0; t < kRows; ++t) p[s][t] = p[s][t] + mine[(s * kRows + t) * 64];
      }
    }
    // strides 32 and 16 of the chunks pair sets, 8 .. 1 lane groups
    f32x4 v;
    if constexpr (NS == 4) v = (p[0] + p[2]) + (p[1] + p[3]);
    else if constexpr (NS == 2) v = p[0] + p[1];
    else v = p[0];
    float ab, cd;
    dm_fold_rows2<32>(v[0], v[1], v[2], v[3], ab, cd);
    float r = dm_fold_rows<16>(ab, cd);
    r = r + dm_xor_lane<8>(r);
    r = r + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, r), 0x124, 0xF, 0xF, false));
    // 16-lane row n holds activation row (0, 2, 1, 3)[n], lane j of it weight row j
    const int t = ((lane >> 5) & 1) | ((lane >> 3) & 2), o = base + kRows * it + j;
    if ((lane & 12) == 0 && ks == 0 && o < O && m0 + t < a.x_rows) {
      const size_t yi = (size_t)(m0 + t) * O + o;
      if (a.y_bf16)
        static_cast<bf16_t*>(sg.y)[yi] = dm_f2bf(r);
      else
        static_cast<float*>(sg.y)[yi] = r;
    }
  }
}

template <int KIND, int NS, int KS, bool XF32>
int go(ornith_ctx* ctx, KqArgs& a, int groups) {
  static const int resident = resident_workgroups(kq_rows_kernel<KIND, NS, KS, XF32>);
  const int asked = a.iters;
  if (!asked) a.iters = auto_iters<16, KS, kRows>(ctx, a, groups, resident);
  const dim3 grid(layout_segments<16, KS>(a), groups);
  hipLaunchKernelGGL((kq_rows_kernel<KIND, NS, KS, XF32>), grid, dim3(256), 0, ctx->stream, a);
  a.iters = asked;
  ORN_LAUNCH_CHECK("kq_rows_kernel");
  return ORNITH_OK;
}
template <int KIND, bool XF32>
int by_width(ornith_ctx* ctx, KqArgs& a, int groups) {
  constexpr bool q4 = KIND == ORNITH_Q4K;
  switch (a.K) {
    case 512: return q4 ? go<ORNITH_Q4K, 1, 1, XF32>(ctx, a, groups) : -1;
    case 1024: return go<KIND, q4 ? 2 : 1, 1, XF32>(ctx, a, groups);
    case 2048: return go<KIND, q4 ? 4 : 2, 1, XF32>(ctx, a, groups);
    case 4096: return go<KIND, q4 ? 4 : 2, 2, XF32>(ctx, a, groups);
    default: return -1;
  }
}

}  // namespace

// Whether a.x_rows activation rows are worth the matrix form: from about 90 million products of a weight
// by a group of four (the measurements above: level at 75 and 100 million, behind it below). Its wavefronts
// hold four weight rows each and need a few steps to pay for the activations' 32 registers a row; smaller
// launches are over in the time of one wavefront's chain, which the matrix instruction (four cycles of its
// own and the wait before it) makes longer.
bool kq_rows_suits(const KqArgs& a) {
  constexpr double kProducts = 9e7;
  long rows = 0;
  for (int i = 0; i < a.nseg; ++i) rows += a.seg[i].O;
  return a.x_rows >= 3 && (double)rows * a.K * ((a.x_rows + kRows - 1) / kRows) >= kProducts;
}

// a.x_rows activation rows in groups of four. -1, nothing launched: a width the kernel does not cover.
int kq_rows(ornith_ctx* ctx, KqArgs& a, int kind, bool x_f32) {
  const int groups = (a.x_rows + kRows - 1) / kRows;
  if (kind == ORNITH_Q4K) return x_f32 ? by_width<ORNITH_Q4K, true>(ctx, a, groups) : by_width<ORNITH_Q4K, false>(ctx, a, groups);
  return x_f32 ? by_width<ORNITH_Q6K, true>(ctx, a, groups) : by_width<ORNITH_Q6K, false>(ctx, a, groups);
}
