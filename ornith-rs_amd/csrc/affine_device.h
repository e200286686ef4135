// Lane-level pieces of the mlx affine mat-vecs: the activation registers of a lane, a row's codes
// with their scales, and a row's contribution to the lane's sums. Shared by the projections
// (affine_mv.hip) and the expert launches (moe_affine4.hip).
//
// The order of a row's sum is affine4_row_dot's / affine8_row_dot's (linear_device.h), whatever the
// launch: lane c of LPR owns the chunks c + LPR i in ascending i (16 codes of the 4-bit group-32
// format, 8 of the 8-bit group-64 one), one fma chain a chunk in code order, scale * chain +
// bias * (sum of the chunk's activations) added to the lane's running value, then the butterfly. A
// row of fewer than 64 chunks leaves the upper lanes of that order at zero, so LPR lanes give its
// bits and a wavefront takes 64 / LPR rows.
#pragma once

#include "dmath.h"

// eight nibbles / four bytes as floats, in code order
__device__ __forceinline__ void a4_codes(uint32_t w, float (&f)[8]) {
  const uint32_t e = w & 0x0f0f0f0fu, o = (w >> 4) & 0x0f0f0f0fu;
  f[0] = dm_ubyte<0>(e); f[1] = dm_ubyte<0>(o);
  f[2] = dm_ubyte<1>(e); f[3] = dm_ubyte<1>(o);
  f[4] = dm_ubyte<2>(e); f[5] = dm_ubyte<2>(o);
  f[6] = dm_ubyte<3>(e); f[7] = dm_ubyte<3>(o);
}

template <int BITS>
struct AffChunk;
template <>
struct AffChunk<4> {
  static constexpr int kCodes = 16, kShift = 1;  // chunks of a scale: 2
};
template <>
struct AffChunk<8> {
  static constexpr int kCodes = 8, kShift = 3;
};

// NC chunks a lane of M activation rows
template <int BITS, int LPR, int NC, int M>
struct AffLane {
  static constexpr int N = AffChunk<BITS>::kCodes;
  float x[M][NC][N], sum[M][NC];
  __device__ __forceinline__ void load(const bf16_t* const (&xr)[M], int c) {
    uint4 raw[M][NC][N / 8];
#pragma unroll
    for (int t = 0; t < M; ++t)
#pragma unroll
      for (int i = 0; i < NC; ++i)
#pragma unroll
        for (int h = 0; h < N / 8; ++h)
          raw[t][i][h] = *reinterpret_cast<const uint4*>(xr[t] + N * (c + LPR * i) + 8 * h);
#pragma unroll
    for (int t = 0; t < M; ++t)
#pragma unroll
      for (int i = 0; i < NC; ++i) {
#pragma unroll
        for (int h = 0; h < N / 8; ++h) {
          const uint32_t w[4] = {raw[t][i][h].x, raw[t][i][h].y, raw[t][i][h].z, raw[t][i][h].w};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            x[t][i][8 * h + 2 * e] = dm_bf2f_lo(w[e]);
            x[t][i][8 * h + 2 * e + 1] = dm_bf2f_hi(w[e]);
          }
        }
        float s = 0.f;
#pragma unroll
        for (int e = 0; e < N; ++e) s = s + x[t][i][e];
        sum[t][i] = s;
      }
  }
};

template <int BITS, int LPR, int NC>
struct AffRow {
  static constexpr int N = AffChunk<BITS>::kCodes;
  uint2 q[NC];
  bf16_t s[NC], b[NC];
  // row `row` of [rows, K] weights, K = N * LPR * NC
  __device__ __forceinline__ void load(const uint8_t* w, const bf16_t* sc, const bf16_t* bi, size_t row, int c) {
    constexpr int CH = LPR * NC, G = CH >> AffChunk<BITS>::kShift;
    const uint8_t* wr = w + row * (8 * CH);
    const bf16_t *sr = sc + row * G, *br = bi + row * G;
#pragma unroll
    for (int i = 0; i < NC; ++i) q[i] = *reinterpret_cast<const uint2*>(wr + 8 * (c + LPR * i));
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      s[i] = sr[(c + LPR * i) >> AffChunk<BITS>::kShift];
      b[i] = br[(c + LPR * i) >> AffChunk<BITS>::kShift];
    }
  }
  // unpacked no earlier than these sums are made (the compiler would unpack every row in hand ahead,
  // 16 registers a chunk)
  template <int M>
  __device__ __forceinline__ void after(const float (&acc)[M]) {
#pragma unroll
    for (int i = 0; i < NC; ++i) asm volatile("" : "+v"(q[i].x), "+v"(q[i].y) : "v"(acc[M - 1]));
  }
  template <int M>
  __device__ __forceinline__ void accumulate(const AffLane<BITS, LPR, NC, M>& L, float (&acc)[M]) const {
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      float f[N];
      if constexpr (BITS == 4) {
        float h[8];
        a4_codes(q[i].x, h);
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = h[e];
        a4_codes(q[i].y, h);
#pragma unroll
        for (int e = 0; e < 8; ++e) f[8 + e] = h[e];
      } else {
        f[0] = dm_ubyte<0>(q[i].x); f[1] = dm_ubyte<1>(q[i].x); f[2] = dm_ubyte<2>(q[i].x); f[3] = dm_ubyte<3>(q[i].x);
        f[4] = dm_ubyte<0>(q[i].y); f[5] = dm_ubyte<1>(q[i].y); f[6] = dm_ubyte<2>(q[i].y); f[7] = dm_ubyte<3>(q[i].y);
      }
      const float sf = dm_bf2f(s[i]), bf = dm_bf2f(b[i]);
#pragma unroll
      for (int t = 0; t < M; ++t) {
        float a = 0.f;
#pragma unroll
        for (int e = 0; e < N; ++e) a = dm_fma(L.x[t][i][e], f[e], a);
        const float p = sf * a;
        acc[t] = acc[t] + dm_fma(L.sum[t][i], bf, p);
      }
    }
  }
};
