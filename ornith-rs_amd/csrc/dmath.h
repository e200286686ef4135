// Device-side scalar arithmetic with fully specified results.
//
// Router indices, argmax tokens and accepted-token counts have to come out the
// same on every run and agree with a scalar CPU evaluation, so nothing here
// calls the device math library: exp/log are written out with fp32 add, mul and
// fma only, divide and sqrt are the correctly rounded IEEE ones (hipcc's
// default), and conversions are integer bit moves or the hardware's exact / round-to-
// nearest-even ones. The file is compiled with -ffp-contract=off, so the only fused
// operations are the explicit __builtin_fmaf.
//
// Rounding points follow the reference: activations are bf16 in memory and fp32
// in registers (/root/reference/kernels/q4k.metal:216-221), bf16 rounding is
// round-to-nearest-even (/root/reference/src/array.rs:229-237).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

typedef uint16_t bf16_t;  // raw bits
typedef uint16_t f16_t;   // raw bits

#define DM_INF (__builtin_inff())

// A pointer rebuilt from an integer that is known to address device memory. Going through the
// global address space lets the compiler use global loads (counted by vmcnt alone, so a kernel
// can wait for its loads one by one) where a bare integer-to-pointer cast gives flat loads.
template <class T>
__device__ __forceinline__ T* dm_global_ptr(uint64_t bits) {
  return (T*)(__attribute__((address_space(1))) T*)bits;
}

// A range of device memory for the buffer loads: what lies past its end reads as zero, so ragged
// blocks need no clamped addresses and no selects. The offset is 32 bits, from a wavefront-wide base; it
// goes into the loads' vector and immediate offsets (the scalar one is not part of the comparison with
// the end, it is taken off the end, which must not wrap).
typedef unsigned int dm_u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int dm_u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t dm_buffer(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}

// p / d for p, d < 2^31, d > 1, with magic = dm_div_magic(d), 2^32 / d rounded up: the upper half of p * magic is the quotient or, from where p times
// what the rounding added passes 2^32, one more.
inline uint32_t dm_div_magic(int d) { return (uint32_t)(((uint64_t(1) << 32) + (uint32_t)d - 1) / (uint32_t)d); }
__device__ __forceinline__ uint32_t dm_div(uint32_t p, uint32_t d, uint32_t magic) {
  const uint32_t q = __umulhi(p, magic);
  return q - (q * d > p ? 1u : 0u);
}

__device__ __forceinline__ float dm_fma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

__device__ __forceinline__ float dm_bf2f(bf16_t b) { return __uint_as_float((uint32_t)b << 16); }

// fp32 -> bf16, round to nearest even: gfx950's v_cvt_pk_bf16_f32 (one instruction for
// two values; subnormals are kept, fp32 denormals being on). Equal to the integer
// formulation u += 0x7fff + ((u >> 16) & 1) for every non-NaN input.
__device__ __forceinline__ bf16_t dm_f2bf(float f) {
  const __bf16 b = (__bf16)f;
  return __builtin_bit_cast(bf16_t, b);
}
// two values in one instruction, element 0 in the low half; each half equals dm_f2bf of its value
__device__ __forceinline__ uint32_t dm_f2bf2(float lo, float hi) {
  typedef float f2v __attribute__((ext_vector_type(2)));
  typedef __bf16 b2v __attribute__((ext_vector_type(2)));
  const f2v v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, b2v));
}
// round to bf16 precision, keep as float
__device__ __forceinline__ float dm_rb(float f) { return dm_bf2f(dm_f2bf(f)); }

// low / high bf16 of a packed pair (little endian: element 0 in the low half)
__device__ __forceinline__ float dm_bf2f_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float dm_bf2f_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

// IEEE half -> float, exact. v_cvt_f32_f16 is exact for every input (subnormals
// included: gfx9 keeps fp16 denormals), so the hardware conversion is used.
__device__ __forceinline__ float dm_h2f(f16_t h) {
  _Float16 v;
  __builtin_memcpy(&v, &h, 2);
  return (float)v;
}

// exp(x): reduce by ln2 in two pieces, degree-5 polynomial, exponent from bits.
// x < -87 gives +0 and x > 88 gives +inf, so subnormal results never occur.
__device__ __forceinline__ float dm_exp(float x) {
  // no branches: the polynomial is worked out for every input and the special cases are
  // selected afterwards (outside [-87, 88] its value is never used; a NaN stays that NaN)
  float n = __builtin_rintf(x * 1.44269504088896341f);
  float r = dm_fma(n, -0.693359375f, x);
  r = dm_fma(n, 2.12194440e-4f, r);
  float p = 1.9875691500e-4f;
  p = dm_fma(p, r, 1.3981999507e-3f);
  p = dm_fma(p, r, 8.3334519073e-3f);
  p = dm_fma(p, r, 4.1665795894e-2f);
  p = dm_fma(p, r, 1.6666665459e-1f);
  p = dm_fma(p, r, 5.0000001201e-1f);
  float r2 = r * r;
  float e = dm_fma(p, r2, r) + 1.0f;
  // n as an integer: n is integral and, where the result is used, within [-126, 127]
  const int ni = (int)__builtin_fminf(__builtin_fmaxf(n, -200.0f), 200.0f);
  float v = e * __uint_as_float((uint32_t)(ni + 127) << 23);
  v = x < -87.0f ? 0.0f : v;
  v = x > 88.0f ? DM_INF : v;
  return x != x ? x : v;
}

// log(x), x finite normal > 0.
__device__ __forceinline__ float dm_log(float x) {
  if (x != x || x < 0.0f) return __builtin_nanf("");
  if (x == 0.0f) return -DM_INF;
  if (x == DM_INF) return DM_INF;
  uint32_t u = __float_as_uint(x);
  int e = (int)(u >> 23) - 126;
  float m = __uint_as_float((u & 0x007fffffu) | 0x3f000000u);
  if (m < 0.707106781186547524f) {
    e -= 1;
    m = m + m;
  }
  float f = m - 1.0f;
  float z = f * f;
  float p = 7.0376836292e-2f;
  p = dm_fma(p, f, -1.1514610310e-1f);
  p = dm_fma(p, f, 1.1676998740e-1f);
  p = dm_fma(p, f, -1.2420140846e-1f);
  p = dm_fma(p, f, 1.4249322787e-1f);
  p = dm_fma(p, f, -1.6668057665e-1f);
  p = dm_fma(p, f, 2.0000714765e-1f);
  p = dm_fma(p, f, -2.4999993993e-1f);
  p = dm_fma(p, f, 3.3333331174e-1f);
  float y = f * z * p;
  float fe = (float)e;
  y = dm_fma(fe, -2.12194440e-4f, y);
  y = dm_fma(-0.5f, z, y);
  float r = f + y;
  r = dm_fma(fe, 0.693359375f, r);
  return r;
}

__device__ __forceinline__ float dm_log1p(float u) {
  float w = 1.0f + u;
  if (w == 1.0f) return u;
  if (w == DM_INF) return DM_INF;
  return dm_log(w) * (u / (w - 1.0f));
}

__device__ __forceinline__ float dm_rsqrt(float x) { return 1.0f / __builtin_sqrtf(x); }

// sigmoid of a bf16 number with every intermediate held in bf16
// (/root/reference/kernels/ornith_sigmoid.h:27-31 at T = bfloat16).
//
// The exponential and the reciprocal are the hardware's: what is kept of each is a bf16, and no
// input brings them within their own error of a rounding boundary. For the reciprocal that follows
// from the numbers: s = a / 2^j with a in [128, 256), and 128 / a is either a power of two or at
// least 2^-18 away from every odd multiple of a half bf16 step. For the exponential, whose argument
// x * log2(e) enters with its rounding error as a second term, it is a matter of the 2^15 inputs
// there are, all of which are compared with the form that dm_exp and a division give
// (tests/test_gpu_kquant.py). 16 vector instructions instead of 50: in the gated-delta front end
// and swiglu at prompt widths the two functions were most of what a channel cost.
__device__ __forceinline__ float dm_sigmoid_bf16(float x) {
  const float a = __builtin_fabsf(x);
  const float t = a * 1.44269504088896341f;
  const float lo = dm_fma(a, 1.925963033e-8f, dm_fma(a, 1.44269504088896341f, -t));
  float e = __builtin_amdgcn_exp2f(t);
  e = dm_fma(e * 0.693147180559945309f, lo, e);
  e = dm_rb(a > 88.0f ? DM_INF : e);
  const float s = dm_rb(1.0f + e);
  // (scaled: the instruction flushes results below the normal range, and 1 / exp(88) is there)
  const float y = dm_rb(__builtin_amdgcn_rcpf(s * 0x1p-32f) * 0x1p-32f);
  return (x < 0.0f) ? y : dm_rb(1.0f - y);
}
// Two at a time with the same bits: the roundings share their instruction.
__device__ __forceinline__ void dm_rb2(float& a, float& b) {
  const uint32_t w = dm_f2bf2(a, b);
  a = dm_bf2f_lo(w);
  b = dm_bf2f_hi(w);
}
__device__ __forceinline__ void dm_sigmoid_bf16x2(float x0, float x1, float& s0, float& s1) {
  const float x[2] = {x0, x1};
  float e[2], s[2], y[2], m[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float a = __builtin_fabsf(x[i]);
    const float t = a * 1.44269504088896341f;
    const float lo = dm_fma(a, 1.925963033e-8f, dm_fma(a, 1.44269504088896341f, -t));
    e[i] = __builtin_amdgcn_exp2f(t);
    e[i] = dm_fma(e[i] * 0.693147180559945309f, lo, e[i]);
    e[i] = a > 88.0f ? DM_INF : e[i];
  }
  dm_rb2(e[0], e[1]);
  for (int i = 0; i < 2; ++i) s[i] = 1.0f + e[i];
  dm_rb2(s[0], s[1]);
  for (int i = 0; i < 2; ++i) y[i] = __builtin_amdgcn_rcpf(s[i] * 0x1p-32f) * 0x1p-32f;
  dm_rb2(y[0], y[1]);
  for (int i = 0; i < 2; ++i) m[i] = 1.0f - y[i];
  dm_rb2(m[0], m[1]);
  s0 = x0 < 0.0f ? y[0] : m[0];
  s1 = x1 < 0.0f ? y[1] : m[1];
}
__device__ __forceinline__ float dm_sigmoid_f32(float x) {
  float y = 1.0f / (1.0f + dm_exp(__builtin_fabsf(x)));
  return (x < 0.0f) ? y : 1.0f - y;
}

// ---- wavefront reductions: v[l] += v[l ^ s], s = 32,16,...,1 ---------------
// fp32 add commutes, so all 64 lanes finish with identical bits.

// Everything here stays in the vector ALU: a trip through the LDS crossbar (ds_swizzle,
// ds_bpermute) costs an LDS round trip each, and a 64-lane sum would take four of them in series.

// The halves of a wavefront (ROWS = 32) or the 16-lane rows of each half (ROWS = 16) trade
// places: given v in both operands, on return a holds the even rows' values in every row pair
// and b the odd rows' (v_permlane32_swap / v_permlane16_swap exchange the odd rows of the
// first operand with the even rows of the second).
template <int ROWS>
__device__ __forceinline__ void dm_row_swap(float v, float& a, float& b) {
  a = v;
  b = v;
  if constexpr (ROWS == 32)
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
  else
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
}

// value of lane (l ^ S): DPP quad permutes for 1 and 2 and a row rotate for 8 (they fold
// into the consuming add), two bank-masked row shifts for 4, a row swap and a select for 16, 32.
template <int S>
__device__ __forceinline__ float dm_xor_lane(float v) {
  int i = __builtin_bit_cast(int, v);
  if constexpr (S == 1)
    i = __builtin_amdgcn_mov_dpp(i, 0xB1, 0xF, 0xF, true);  // quad_perm [1,0,3,2]
  else if constexpr (S == 2)
    i = __builtin_amdgcn_mov_dpp(i, 0x4E, 0xF, 0xF, true);  // quad_perm [2,3,0,1]
  else if constexpr (S == 4) {
    const int up = __builtin_amdgcn_update_dpp(i, i, 0x104, 0xF, 0x5, false);  // row_shl:4 into lanes 0-3, 8-11
    i = __builtin_amdgcn_update_dpp(up, i, 0x114, 0xF, 0xA, false);            // row_shr:4 into lanes 4-7, 12-15
  } else if constexpr (S == 8)
    i = __builtin_amdgcn_update_dpp(0, i, 0x128, 0xF, 0xF, false);  // row_ror:8 (every lane has a source)
  else {
    float a, b;
    dm_row_swap<S>(v, a, b);
    return (__lane_id() & S) ? a : b;
  }
  return __builtin_bit_cast(float, i);
}

template <int WIDTH>
__device__ __forceinline__ float dm_wave_sum(float v) {
  // a + b after a row swap is v[l] + v[l ^ ROWS] with the operands in one order for both
  // partners, which is the same bits
  if constexpr (WIDTH >= 64) { float a, b; dm_row_swap<32>(v, a, b); v = a + b; }
  if constexpr (WIDTH >= 32) { float a, b; dm_row_swap<16>(v, a, b); v = a + b; }
  if constexpr (WIDTH >= 16) {
    v = v + dm_xor_lane<8>(v);
    // v now repeats every 8 lanes, so the lane 4 further round the row holds the bits of lane
    // l ^ 4: one rotate that folds into the add
    v = v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x124, 0xF, 0xF, false));
  } else if constexpr (WIDTH >= 8) {
    v = v + dm_xor_lane<4>(v);
  }
  if constexpr (WIDTH >= 4) v = v + dm_xor_lane<2>(v);
  if constexpr (WIDTH >= 2) v = v + dm_xor_lane<1>(v);
  return v;
}
template <int WIDTH>
__device__ __forceinline__ float dm_wave_max(float v) {
  float o;
  if constexpr (WIDTH >= 64) { float a, b; dm_row_swap<32>(v, a, b); v = b > a ? b : a; }
  if constexpr (WIDTH >= 32) { float a, b; dm_row_swap<16>(v, a, b); v = b > a ? b : a; }
  if constexpr (WIDTH >= 16) { o = dm_xor_lane<8>(v); v = o > v ? o : v; }
  if constexpr (WIDTH >= 8) { o = dm_xor_lane<4>(v); v = o > v ? o : v; }
  if constexpr (WIDTH >= 4) { o = dm_xor_lane<2>(v); v = o > v ? o : v; }
  if constexpr (WIDTH >= 2) { o = dm_xor_lane<1>(v); v = o > v ? o : v; }
  return v;
}

// Several butterfly sums for the price of one and a bit. A swap of rows between TWO values leaves in
// their sum the first one's pair in the even rows and the second one's in the odd rows, so the 32 and
// 16 steps (and, with a select, the 8 step) halve the number of values instead of repeating them.
// Every addition pairs the same two operands as the plain butterfly, so the bits are those of
// dm_wave_sum.
template <int ROWS>
__device__ __forceinline__ float dm_fold_rows(float a, float b) {
  if constexpr (ROWS == 32)
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
  else
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
  return a + b;
}
// two pairs, the waits shared
template <int ROWS>
__device__ __forceinline__ void dm_fold_rows2(float a, float b, float c, float d, float& ab, float& cd) {
  if constexpr (ROWS == 32)
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\tv_permlane32_swap_b32 %2, %3\n\ts_nop 1" : "+v"(a), "+v"(b), "+v"(c), "+v"(d));
  else
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\tv_permlane16_swap_b32 %2, %3\n\ts_nop 1" : "+v"(a), "+v"(b), "+v"(c), "+v"(d));
  ab = a + b;
  cd = c + d;
}
// the steps 8 .. 1 of a butterfly: lane l ends with the sum over its row of 16
__device__ __forceinline__ float dm_row_sum(float v) {
  v = v + dm_xor_lane<8>(v);
  v = v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x124, 0xF, 0xF, false));
  v = v + dm_xor_lane<2>(v);
  return v + dm_xor_lane<1>(v);
}
// Four 64-lane sums: on return lanes [0,16) hold sum(a), [16,32) sum(c), [32,48) sum(b), [48,64) sum(d).
__device__ __forceinline__ float dm_wave_sum4(float a, float b, float c, float d) {
  float ab, cd;
  dm_fold_rows2<32>(a, b, c, d, ab, cd);
  return dm_row_sum(dm_fold_rows<16>(ab, cd));
}
// M sums over groups of W lanes, one of them in each of the lanes for which dm_multi_leads holds:
// lane c of the group has sum dm_multi_of(c) of them (>= M: none).
template <int W, int M>
__device__ __forceinline__ float dm_multi_sum(const float (&v)[M]) {
  if constexpr (M == 1 || W < 32) {
    static_assert(M == 1, "groups of 32 or 64 lanes");
    return dm_wave_sum<W>(v[0]);
  } else if constexpr (W == 64) {
    if constexpr (M == 2) {
      float a, b, r = dm_fold_rows<32>(v[0], v[1]);
      dm_row_swap<16>(r, a, b);
      return dm_row_sum(a + b);
    } else {
      return dm_wave_sum4(v[0], v[1], v[2], M > 3 ? v[M - 1] : 0.f);
    }
  } else {
    if constexpr (M == 2) {
      return dm_row_sum(dm_fold_rows<16>(v[0], v[1]));
    } else {
      float ab, cd;
      dm_fold_rows2<16>(v[0], v[1], v[2], M > 3 ? v[M - 1] : 0.f, ab, cd);
      const bool h8 = __lane_id() & 8;
      float r = (h8 ? cd : ab) + dm_xor_lane<8>(h8 ? ab : cd);
      r = r + dm_xor_lane<4>(r);
      r = r + dm_xor_lane<2>(r);
      return r + dm_xor_lane<1>(r);
    }
  }
}
template <int W, int M>
__device__ __forceinline__ bool dm_multi_leads(int c) {
  return (c & ((M == 1 ? W : M == 2 ? W / 2 : W / 4) - 1)) == 0;
}
template <int W, int M>
__device__ __forceinline__ int dm_multi_of(int c) {
  return M == 1 ? 0 : M == 2 ? c / (W / 2) : (c / (W / 2)) | (c / (W / 4) & 1) << 1;
}
__device__ __forceinline__ float dm_lane_value(float v, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

// Fused multiply-adds whose first factor is one lane's value of a 16-lane row (DPP row_newbcast): a
// factor that is the same for all lanes, a query's channels or a row of probabilities, stays one
// value a lane, 16 to a register in every row, and is neither read from LDS nor moved to a scalar
// register for each use (a 16-byte broadcast read is 16 clocks of the compute unit's LDS, a
// v_readlane the price of the multiply-add). All 64 lanes must be active. The two wait states that a
// DPP read needs after its register was written stand at the head of each group.
#define DM_FMAC(A, X, Y, I) "v_fmac_f32_dpp %" #A ", %" #X ", %" #Y " row_newbcast:" #I " row_mask:0xf bank_mask:0xf\n\t"
// acc[j] += q[j](lane B + e) * k[e], e = 0 .. 7 in order, B = 0 or 8
template <int B>
__device__ __forceinline__ void dm_dot8(float& a, float q, const float (&k)[8]) {
  if constexpr (B == 0)
    asm("s_nop 1\n\t" DM_FMAC(0, 1, 2, 0) DM_FMAC(0, 1, 3, 1) DM_FMAC(0, 1, 4, 2) DM_FMAC(0, 1, 5, 3) DM_FMAC(0, 1, 6, 4)
            DM_FMAC(0, 1, 7, 5) DM_FMAC(0, 1, 8, 6) DM_FMAC(0, 1, 9, 7)
        : "+&v"(a)
        : "v"(q), "v"(k[0]), "v"(k[1]), "v"(k[2]), "v"(k[3]), "v"(k[4]), "v"(k[5]), "v"(k[6]), "v"(k[7]));
  else
    asm("s_nop 1\n\t" DM_FMAC(0, 1, 2, 8) DM_FMAC(0, 1, 3, 9) DM_FMAC(0, 1, 4, 10) DM_FMAC(0, 1, 5, 11) DM_FMAC(0, 1, 6, 12)
            DM_FMAC(0, 1, 7, 13) DM_FMAC(0, 1, 8, 14) DM_FMAC(0, 1, 9, 15)
        : "+&v"(a)
        : "v"(q), "v"(k[0]), "v"(k[1]), "v"(k[2]), "v"(k[3]), "v"(k[4]), "v"(k[5]), "v"(k[6]), "v"(k[7]));
}
// o[e] += w(lane B + u) * v[u][e], u = 0 .. 3 in order: two channels, four keys; B = 0, 4, 8, 12
#define DM_FMACW(V0, V1, I) DM_FMAC(0, 2, V0, I) DM_FMAC(1, 2, V1, I)
#define DM_AXPY2(I0, I1, I2, I3)                                                                                          \
  asm("s_nop 1\n\t" DM_FMACW(3, 4, I0) DM_FMACW(5, 6, I1) DM_FMACW(7, 8, I2) DM_FMACW(9, 10, I3)                           \
      : "+&v"(o[0]), "+&v"(o[1])                                                                                            \
      : "v"(w), "v"(v[0][0]), "v"(v[0][1]), "v"(v[1][0]), "v"(v[1][1]), "v"(v[2][0]), "v"(v[2][1]), "v"(v[3][0]), "v"(v[3][1]))
template <int B>
__device__ __forceinline__ void dm_axpy4(float (&o)[2], float w, const float (&v)[4][2]) {
  if constexpr (B == 0) DM_AXPY2(0, 1, 2, 3);
  else if constexpr (B == 4) DM_AXPY2(4, 5, 6, 7);
  else if constexpr (B == 8) DM_AXPY2(8, 9, 10, 11);
  else DM_AXPY2(12, 13, 14, 15);
}
#undef DM_FMACW
#undef DM_AXPY2
#undef DM_FMAC

// byte k of a dword as a float, one instruction (the compiler's own pattern match gives
// a bit-field extract plus a convert once the operand carries a nibble mask)
__device__ __forceinline__ float dm_ubyte0(uint32_t w) { float r; asm("v_cvt_f32_ubyte0 %0, %1" : "=v"(r) : "v"(w)); return r; }
__device__ __forceinline__ float dm_ubyte1(uint32_t w) { float r; asm("v_cvt_f32_ubyte1 %0, %1" : "=v"(r) : "v"(w)); return r; }
__device__ __forceinline__ float dm_ubyte2(uint32_t w) { float r; asm("v_cvt_f32_ubyte2 %0, %1" : "=v"(r) : "v"(w)); return r; }
__device__ __forceinline__ float dm_ubyte3(uint32_t w) { float r; asm("v_cvt_f32_ubyte3 %0, %1" : "=v"(r) : "v"(w)); return r; }
template <int K>
__device__ __forceinline__ float dm_ubyte(uint32_t w) {
  if constexpr (K == 0) return dm_ubyte0(w);
  else if constexpr (K == 1) return dm_ubyte1(w);
  else if constexpr (K == 2) return dm_ubyte2(w);
  else return dm_ubyte3(w);
}
