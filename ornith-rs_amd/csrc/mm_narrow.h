// GEMM of few activation rows over quantized weights (prompts of some tens to some hundreds of
// tokens, and the routed experts of longer ones): Y[M, O] = X[M, K] . W^T on the matrix cores,
// plain or over an expert-sorted pair list, and the expert form with gate, up and swiglu in one.
//
// What bounds these calls is not arithmetic: a 51-row projection of 12288 x 2048 is 2.6 GFLOP
// over 14 MB, an expert has 2 to 40 rows. The wide kernels of kq_mm.hip walk K in slabs with a
// barrier each, one 128-column block a workgroup: 16 slabs of load -> dequantize -> barrier ->
// MFMA in series, on 96 (or, for a 512-column projection, 4) of 256 compute units, 43 us for that
// projection. Here a workgroup's wavefronts split K instead: each has the weights of its 256-wide K
// block for 16 * CT columns in flight at once, straight into registers, turns them into MFMA operands
// there (v_mfma_f32_16x16x32_bf16: a lane supplies eight consecutive k of one weight row), and the
// partial tiles meet in LDS once. No barrier inside the K loop, and narrow projections become O / 16
// workgroups.
//
// What such a kernel can run against is the L1's tag lookups: 64 lanes that each read their own row
// are 64 lookups a load instruction, one a clock and compute unit, whatever a lane takes. So every lane
// takes 16 bytes of codes a load, the activations come in as whole 64- or 128-byte pieces of a row straight
// into LDS (global_load_lds: no registers; each wavefront its own K block, so nothing waits for another
// wavefront), and the scales of all the workgroup's rows, which lie side by side in memory, as one
// block. The k order inside a block is free as long as both operands follow it, and is chosen so that
// 16 bytes of codes make a lane's operands (piece()).
//
// Counters of the expert launches: 28 to 39 lookups a load instruction and the L1
// busy 35 to 42 % of the time, the matrix cores 5 to 14 %, the vector units 48 to 66 % (the codes' way to
// operands), 3.6 to 4.1 TB/s from memory: vector issue beside the stream is what bounds them. The
// plain launches of a short prompt are one pass of a chain: load, unpack, multiply, meet (vector units 13 %).
//
// Measured (us, before -> now): 12288 x 2048 Q4_K at 64 rows 29.5 -> 15.8, 2048 x 4096 at 64 rows 52 -> 11.8,
// 256 x 2048 Q6_K 28.6 -> 7.1; the experts of a 51-token prompt, gate + up + swiglu 104 -> 54 (193 MB from memory),
// down 49 -> 36.5 (142 MB), of a 700-token one 156 -> 122 and 76 -> 82 (the shared expert included); a
// 600-token prompt over 4-bit affine weights 461 ms -> 15.9 ms (its experts and projections were mat-vecs,
// row by row).
//
// The order of the sums depends on K alone (256-wide blocks: wavefront ks takes blocks ks, ks + KS,
// ...; the partial sums are added in one order), never on M, O or the launch's other matrices.
//
// Weight formats:
//   Q4_K, Q6_K        dequantized with kquant::dequantize's arithmetic and rounded to bf16, as in
//                     kq_mm.hip
//   affine 4 / 8 bit  the codes are exact bf16 numbers and go to the matrix cores as they are; the
//                     sum over a group (32 / 64 k, one / two MFMAs) is multiplied by the group's
//                     scale in fp32, and the bias meets the group's sum of activations, which the
//                     same matrix core makes from a column of ones. No weight is rounded: the
//                     arithmetic is that of the mat-vec (linear.hip), summed in another order.
#pragma once

#include <type_traits>

#include "dmath.h"
#include "moe_device.h"
#include "rt.h"

namespace nmm {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));

enum Kind { kQ4K = 0, kQ6K = 1, kA4 = 2, kA8 = 3 };
enum Mode { kPlain = 0, kGather = 1, kGateUp = 2 };

struct Mat {
  const uint8_t* q;  // codes
  const uint8_t* s;  // k-quant scales; affine scales (bf16)
  const uint8_t* d;  // k-quant d (and dmin); affine biases (bf16)
  bf16_t* y;
  int O, kind;
  int cb0;  // plain form: first column block of the launch that is this matrix's
};

struct Args {
  Mat m[4];  // plain: up to four matrices; gathered: [0] routed (or gate), [1] routed up, [2] shared (gate), [3] shared up
  int n;
  const bf16_t* x;
  int M, K, ks;  // ks: wavefronts that split K (2 or 4)
  // gathered forms: tiles over (expert, row range) of an expert-sorted pair list. Expert E is the
  // shared one: its "pairs" are pairs + token.
  const uint32_t* pair;
  const uint32_t* tile_expert;
  const uint32_t* tile_start;
  const uint32_t* tile_count;
  const uint32_t* n_tiles;
  int up_div, pairs, E;
};

// bytes of a 256-weight block in the three tensors
__host__ __device__ constexpr int q_bytes(int kind) { return kind == kQ6K ? 192 : kind == kA8 ? 256 : 128; }
__host__ __device__ constexpr int s_bytes(int kind) { return kind == kQ4K ? 12 : kind == kA8 ? 8 : 16; }
__host__ __device__ constexpr int d_bytes(int kind) { return kind == kQ4K ? 4 : kind == kQ6K ? 2 : kind == kA4 ? 16 : 8; }

// A base the whole wavefront shares (scalar registers) and a lane's 32-bit offset. The offset is made
// opaque where it is used: hoisted out of the K loop it would become a 64-bit register pair a load,
// and the spills of those wait for every load in flight.
template <class V>
__device__ __forceinline__ V ld_off(const uint8_t* base, uint32_t off) {
  asm volatile("" : "+v"(off));
  return *reinterpret_cast<const V*>(base + off);
}
// 16 bytes a lane from memory to LDS: the wavefront's 64 pieces land side by side at `lds`
__device__ __forceinline__ void dma16(const uint8_t* base, uint32_t off, uint32_t lds) {
  asm volatile("" : "+v"(off));
  typedef const __attribute__((address_space(1))) void glb_t;
  typedef __attribute__((address_space(3))) void lds_t;
  __builtin_amdgcn_global_load_lds((glb_t*)(uint64_t)(base + off), (lds_t*)(uint64_t)lds, 16, 0, 0);
}
// a pointer every lane of the wavefront holds alike, in scalar registers
__device__ __forceinline__ const uint8_t* uniform(const uint8_t* p) {
  const uint64_t v = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return dm_global_ptr<const uint8_t>(((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return (uint32_t)(uint64_t)(const __attribute__((address_space(3))) void*)p;
}
// (the compiler does not connect LDS reads with the loads that filled it: the waits are written out)
template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// ---- weight tiles: 16 weight rows x 256 k, lane (c = lane & 15, q = lane >> 4) ------------------
// A block is eight k steps of 32, two to an activation chunk u. A chunk row has eight 16-byte slots of
// eight k: lane q reads slot<H>(q) for step 2 u + H, and slot s of chunk u is piece(u, s) of the block's
// 32 (k = 8 * piece ..).
//   frag<S>()  the lane's operand of step S, from load()'s registers and scales<U>()'s
template <int KIND>
struct Tile;

__device__ __forceinline__ bf16x8_t as_frag(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  const u32x4_t v = {a, b, c, d};
  return __builtin_bit_cast(bf16x8_t, v);
}
// w = s * code + o of eight codes (bytes), rounded to bf16
__device__ __forceinline__ bf16x8_t scaled(uint32_t c0, uint32_t c1, float s, float o) {
  return as_frag(dm_f2bf2(dm_fma(s, dm_ubyte<0>(c0), o), dm_fma(s, dm_ubyte<1>(c0), o)),
                 dm_f2bf2(dm_fma(s, dm_ubyte<2>(c0), o), dm_fma(s, dm_ubyte<3>(c0), o)),
                 dm_f2bf2(dm_fma(s, dm_ubyte<0>(c1), o), dm_fma(s, dm_ubyte<1>(c1), o)),
                 dm_f2bf2(dm_fma(s, dm_ubyte<2>(c1), o), dm_fma(s, dm_ubyte<3>(c1), o)));
}

// Q4_K: lane q takes pieces q (steps 0 - 3) and q + 4 of the block's eight 16-byte code pieces; piece
// p is bytes 16 (p & 1) .. of 64-group p >> 1, low nibbles k = 64 (p >> 1) + 16 (p & 1) + i, high
// ones 32 further on. Chunk u = (half, nibble).
template <>
struct Tile<kQ4K> {
  static constexpr bool kAffine = false;
  static constexpr int kSteps = 1;
  u32x4_t w[2];
  float s, o;
  static __device__ __forceinline__ int piece(int u, int slot) {
    return 16 * (u >> 1) + 4 * (u & 1) + 8 * (slot >> 2) + (slot & 3);
  }
  template <int H>
  static __device__ __forceinline__ int slot(int q) { return 2 * q + H; }
  __device__ __forceinline__ void load(const uint8_t* cq, uint32_t blk, int q) {
    w[0] = ld_off<u32x4_t>(cq, blk * q_bytes(kQ4K) + 16 * q);
    w[1] = ld_off<u32x4_t>(cq + 64, blk * q_bytes(kQ4K) + 16 * q);
  }
  // sub-block 4 (u >> 1) + 2 (q >> 1) + (u & 1) of the block whose scales are at ls / ld in LDS
  template <int U>
  __device__ __forceinline__ void scales(const uint8_t* ls, const uint8_t* ld, int q) {
    const uint32_t* sc = reinterpret_cast<const uint32_t*>(ls);
    const int sh = 16 * (q >> 1) + 8 * (U & 1);
    uint32_t sb, mb;
    if constexpr (U < 2) {
      sb = (sc[0] >> sh) & 63u;
      mb = (sc[1] >> sh) & 63u;
    } else {
      const uint32_t t = sc[2] >> sh;
      sb = (t & 15u) | (((sc[0] >> sh) >> 2) & 0x30u);
      mb = ((t >> 4) & 15u) | (((sc[1] >> sh) >> 2) & 0x30u);
    }
    const uint32_t dmw = *reinterpret_cast<const uint32_t*>(ld);
    s = dm_h2f((f16_t)(dmw & 0xffffu)) * (float)sb;
    o = -(dm_h2f((f16_t)(dmw >> 16)) * (float)mb);
  }
  template <int S>
  __device__ __forceinline__ bf16x8_t frag() const {
    constexpr int NIB = (S >> 1) & 1, W = 2 * (S & 1);
    return scaled((w[S >> 2][W] >> (4 * NIB)) & 0x0f0f0f0fu, (w[S >> 2][W + 1] >> (4 * NIB)) & 0x0f0f0f0fu, s, o);
  }
};

// Q6_K: lane q takes positions 16 (q & 1) .. of the 128-half q >> 1: 16 bytes of each of the half's
// two low-nibble rows and of its high bits. Chunk u = quarter of the halves (k = 128 half + 32 u + position).
template <>
struct Tile<kQ6K> {
  static constexpr bool kAffine = false;
  static constexpr int kSteps = 1;
  u32x4_t la, lb, h;
  float s, o;
  static __device__ __forceinline__ int piece(int u, int slot) { return 16 * (slot >> 2) + 4 * u + (slot & 3); }
  template <int H>
  static __device__ __forceinline__ int slot(int q) { return 2 * q + H; }
  __device__ __forceinline__ void load(const uint8_t* cq, uint32_t blk, int q) {
    const uint32_t at = blk * q_bytes(kQ6K) + 64 * (q >> 1) + 16 * (q & 1);
    la = ld_off<u32x4_t>(cq, at);
    lb = ld_off<u32x4_t>(cq + 32, at);
    h = ld_off<u32x4_t>(cq + 128, blk * q_bytes(kQ6K) + 16 * q);
  }
  // scale 8 (q >> 1) + 2 u + (q & 1) of the block's sixteen
  template <int U>
  __device__ __forceinline__ void scales(const uint8_t* ls, const uint8_t* ld, int q) {
    const int8_t sc = (int8_t)ls[8 * (q >> 1) + 2 * U + (q & 1)];
    s = dm_h2f(*reinterpret_cast<const f16_t*>(ld)) * (float)(int)sc;
    o = -32.f * s;
  }
  template <int S>
  __device__ __forceinline__ bf16x8_t frag() const {
    constexpr int QD = S >> 1, NIB = QD >> 1, W = 2 * (S & 1);
    const u32x4_t& lo = (QD & 1) ? lb : la;
    return scaled(((lo[W] >> (4 * NIB)) & 0x0f0f0f0fu) | (((h[W] >> (2 * QD)) & 0x03030303u) << 4),
                  ((lo[W + 1] >> (4 * NIB)) & 0x0f0f0f0fu) | (((h[W + 1] >> (2 * QD)) & 0x03030303u) << 4), s, o);
  }
};

// byte 0000nnnn as an 8-bit float (4 exponent bits, 3 mantissa bits) is exactly n * 2^-9, so the
// scaled conversion with 2^9 gives the bf16 number n: two codes an instruction
__device__ __forceinline__ uint32_t code_pair(uint32_t w, bool hi) {
  typedef __bf16 b2v __attribute__((ext_vector_type(2)));
  const b2v v = hi ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 512.0f, true)
                   : __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 512.0f, false);
  return __builtin_bit_cast(uint32_t, v);
}
// the odd 16-lane rows of a trade places with the even ones of b (ROWS = 16), or the upper half
// of a with the lower half of b (ROWS = 32)
template <int ROWS>
__device__ __forceinline__ void swap_rows(uint32_t& a, uint32_t& b) {
  if constexpr (ROWS == 32)
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
  else
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
}

// 4-bit affine: a step is one group of 32 (its scale is applied to the step's products, so the four
// lanes of a column have to be in the same group): natural k order.
template <>
struct Tile<kA4> {
  static constexpr bool kAffine = true;
  static constexpr int kSteps = 1;  // k steps a group
  u32x4_t t[2];                     // word q of groups 4 i + g
  u32x4_t sc, bi;                   // the block's eight scales and biases, two to a word
  static __device__ __forceinline__ int piece(int u, int slot) { return 8 * u + slot; }
  template <int H>
  static __device__ __forceinline__ int slot(int q) { return 4 * H + q; }
  __device__ __forceinline__ void load(const uint8_t* cq, uint32_t blk, int q) {
    // whole groups (16 bytes): lane q holds group 4 i + q
    t[0] = ld_off<u32x4_t>(cq, blk * q_bytes(kA4) + 16 * q);
    t[1] = ld_off<u32x4_t>(cq + 64, blk * q_bytes(kA4) + 16 * q);
  }
  // word g of group q -> word q of group g: the 4 x 4 transpose over the lanes of a column
  template <int I>
  __device__ __forceinline__ void transpose() {
    uint32_t a = t[I][0], b = t[I][1], c = t[I][2], d = t[I][3];
    swap_rows<32>(a, c);
    swap_rows<32>(b, d);
    swap_rows<16>(a, b);
    swap_rows<16>(c, d);
    t[I] = u32x4_t{a, b, c, d};
  }
  template <int U>
  __device__ __forceinline__ void scales(const uint8_t* ls, const uint8_t* ld, int) {
    if constexpr (U == 0) {
      transpose<0>();
      sc = *reinterpret_cast<const u32x4_t*>(ls);
      bi = *reinterpret_cast<const u32x4_t*>(ld);
    }
    if constexpr (U == 2) transpose<1>();
  }
  template <int S>
  __device__ __forceinline__ float scale() const { return (S & 1) ? dm_bf2f_hi(sc[S >> 1]) : dm_bf2f_lo(sc[S >> 1]); }
  template <int S>
  __device__ __forceinline__ float bias() const { return (S & 1) ? dm_bf2f_hi(bi[S >> 1]) : dm_bf2f_lo(bi[S >> 1]); }
  template <int S>
  __device__ __forceinline__ bf16x8_t frag() const {
    const uint32_t w = t[S >> 2][S & 3];
    const uint32_t even = w & 0x0f0f0f0fu, odd = (w >> 4) & 0x0f0f0f0fu;
    // codes 0 1 2 3 and 4 5 6 7 as bytes
    const uint32_t a = __builtin_amdgcn_perm(odd, even, 0x05010400u), b = __builtin_amdgcn_perm(odd, even, 0x07030602u);
    return as_frag(code_pair(a, false), code_pair(a, true), code_pair(b, false), code_pair(b, true));
  }
};

// 8-bit affine: a chunk is one group of 64, natural k order
template <>
struct Tile<kA8> {
  static constexpr bool kAffine = true;
  static constexpr int kSteps = 2;
  u32x2_t w[8];
  u32x2_t sc, bi;  // the block's four scales and biases
  static __device__ __forceinline__ int piece(int u, int slot) { return 8 * u + slot; }
  template <int H>
  static __device__ __forceinline__ int slot(int q) { return 4 * H + q; }
  __device__ __forceinline__ void load(const uint8_t* cq, uint32_t blk, int q) {
#pragma unroll
    for (int i = 0; i < 8; ++i) w[i] = ld_off<u32x2_t>(cq + 32 * i, blk * q_bytes(kA8) + 8 * q);
  }
  template <int U>
  __device__ __forceinline__ void scales(const uint8_t* ls, const uint8_t* ld, int) {
    if constexpr (U == 0) {
      sc = *reinterpret_cast<const u32x2_t*>(ls);
      bi = *reinterpret_cast<const u32x2_t*>(ld);
    }
  }
  template <int S>
  __device__ __forceinline__ float scale() const { return (S & 2) ? dm_bf2f_hi(sc[S >> 2]) : dm_bf2f_lo(sc[S >> 2]); }
  template <int S>
  __device__ __forceinline__ float bias() const { return (S & 2) ? dm_bf2f_hi(bi[S >> 2]) : dm_bf2f_lo(bi[S >> 2]); }
  template <int S>
  __device__ __forceinline__ bf16x8_t frag() const {  // 0 .. 255 are bf16 numbers
    const uint32_t a = w[S][0], b = w[S][1];
    return as_frag(dm_f2bf2(dm_ubyte<0>(a), dm_ubyte<1>(a)), dm_f2bf2(dm_ubyte<2>(a), dm_ubyte<3>(a)),
                   dm_f2bf2(dm_ubyte<0>(b), dm_ubyte<1>(b)), dm_f2bf2(dm_ubyte<2>(b), dm_ubyte<3>(b)));
  }
};

// ---- one wavefront's share: RT x CT tiles of 16 x 16 over its K blocks ----------------------------
// NB: activation chunks (2 KB * RT each) its part of LDS holds
template <int KIND, int RT, int CT, int NB>
struct Work {
  typedef Tile<KIND> T;
  f32x4_t acc[RT][CT];
  T t[CT];
  uint32_t ls0, ld0;      // LDS offsets of the scales of the lane's row of tile 0
  uint32_t ls_[CT], ld_[CT];  // ... of the other tiles from there (the same for every lane)

  // chunk U of the block at x into buffer U % NB: a row's eight slots lie permuted (slot s at
  // s ^ (row & 7)), so that the 16 rows a fragment read takes a slot from are on different banks
  template <int U>
  __device__ __forceinline__ void fetch(const uint8_t* x, const uint32_t (&xo)[2 * RT], uint32_t lds, int lane) const {
    const uint32_t p = 16 * (uint32_t)T::piece(U, (lane & 7) ^ (lane >> 3));
#pragma unroll
    for (int i = 0; i < 2 * RT; ++i) dma16(x, xo[i] + p, lds + (U % NB) * (RT * 2048) + i * 1024);
  }
  template <int S>
  __device__ __forceinline__ void step(const uint8_t* smem, const uint8_t* xs, int c, int q) {
    constexpr int U = S >> 1, H = S & 1;
    bf16x8_t a[RT];
    auto read = [&](auto hc, bf16x8_t (&dst)[RT]) {
      constexpr int HH = decltype(hc)::value;
      const uint8_t* p = xs + (U % NB) * (RT * 2048) + c * 128 + 16 * (T::template slot<HH>(q) ^ (c & 7));
#pragma unroll
      for (int r = 0; r < RT; ++r) dst[r] = *reinterpret_cast<const bf16x8_t*>(p + r * 2048);
    };
    if constexpr (!T::kAffine) {
      read(std::integral_constant<int, H>{}, a);
#pragma unroll
      for (int j = 0; j < CT; ++j) {
        if constexpr (H == 0) t[j].template scales<U>(smem + ls0 + ls_[j], smem + ld0 + ld_[j], q);
        const bf16x8_t b = t[j].template frag<S>();
#pragma unroll
        for (int r = 0; r < RT; ++r) acc[r][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[r], b, acc[r][j], 0, 0, 0);
      }
    } else if constexpr (S % T::kSteps == 0) {
      constexpr int N = T::kSteps;
      const bf16x8_t ones = as_frag(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u);
      const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
      bf16x8_t a1[RT];
      f32x4_t sx[RT];  // the rows' sums over the group, in every column
      read(std::integral_constant<int, H>{}, a);
      if constexpr (N == 2) read(std::integral_constant<int, 1>{}, a1);
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        sx[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[r], ones, zero, 0, 0, 0);
        if constexpr (N == 2) sx[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1[r], ones, sx[r], 0, 0, 0);
      }
#pragma unroll
      for (int j = 0; j < CT; ++j) {
        if constexpr (H == 0) t[j].template scales<U>(smem + ls0 + ls_[j], smem + ld0 + ld_[j], q);
        const bf16x8_t b = t[j].template frag<S>();
        f32x4_t g[RT];
#pragma unroll
        for (int r = 0; r < RT; ++r) g[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[r], b, zero, 0, 0, 0);
        if constexpr (N == 2) {
          const bf16x8_t b1 = t[j].template frag<(S + N - 1)>();
#pragma unroll
          for (int r = 0; r < RT; ++r) g[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1[r], b1, g[r], 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            acc[r][j][e] = dm_fma(t[j].template scale<S>(), g[r][e], dm_fma(t[j].template bias<S>(), sx[r][e], acc[r][j][e]));
      }
    }
    // (or the scheduler dequantizes the whole block ahead, and spills)
    __builtin_amdgcn_sched_barrier(0);
  }
  // x, xo: the activations and the byte offsets of the rows this lane fetches; code: the two halves'
  // codes (GC column tiles each); row0: the lane's weight row of tile 0, O: their number; xs / lds:
  // this wavefront's activation buffers; first(): what has to be done before the first block's arithmetic
  template <int GC, class F>
  __device__ __forceinline__ void run(const uint8_t* const (&code)[2], int row0, int O, const bf16_t* x,
                                      const uint32_t (&xo)[2 * RT], int nb, int ks, int KS, int lane, const uint8_t* smem,
                                      const uint8_t* xs, uint32_t lds, F first) {
    const int c = lane & 15, q = lane >> 4;
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int j = 0; j < CT; ++j) acc[r][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int ib = ks; ib < nb; ib += KS) {
      const uint8_t* xk = reinterpret_cast<const uint8_t*>(x) + (size_t)ib * 512;
      fetch<0>(xk, xo, lds, lane);
      fetch<1>(xk, xo, lds, lane);
      if constexpr (NB == 4) {
        fetch<2>(xk, xo, lds, lane);
        fetch<3>(xk, xo, lds, lane);
      }
#pragma unroll
      for (int j = 0; j < CT; ++j) t[j].load(code[j / GC] + (size_t)ib * q_bytes(KIND), (uint32_t)min(row0 + 16 * (j % GC), O - 1) * (uint32_t)nb, q);
      wait_loads<0>();
      if (ib == ks) first();
      step<0>(smem, xs, c, q);
      step<1>(smem, xs, c, q);
      if constexpr (NB == 2) fetch<2>(xk, xo, lds, lane);
      step<2>(smem, xs, c, q);
      step<3>(smem, xs, c, q);
      if constexpr (NB == 2) {
        fetch<3>(xk, xo, lds, lane);
        wait_loads<2 * RT>();
      }
      step<4>(smem, xs, c, q);
      step<5>(smem, xs, c, q);
      if constexpr (NB == 2) wait_loads<0>();
      step<6>(smem, xs, c, q);
      step<7>(smem, xs, c, q);
      ls0 += KS * s_bytes(KIND);
      ld0 += KS * d_bytes(KIND);
    }
  }
};

constexpr int kLdsBytes = 160 * 1024;
constexpr int kPad = 4;  // a row of a partial tile: 16 CT + 4 floats, so the four 4-row groups of a store hit other banks

// LDS of a workgroup: activation chunks of its NW wavefronts, then the scales of its rows; the
// partial tiles go over both (host and device share the arithmetic)
__host__ __device__ constexpr int chunks_held(int rows) { return rows <= 16 ? 4 : 2; }
__host__ __device__ constexpr int x_bytes(int rows, int nw) { return nw * chunks_held(rows) * (rows / 16) * 2048; }
__host__ __device__ constexpr int red_bytes(int rows, int ct, int nw) { return nw / 2 * rows * (16 * ct + kPad) * 4; }

// a workgroup's tile of up to 16 RT rows: partial products, their sums, the outputs
template <int KIND, int RT, int CT, int MODE, int ROWS, int NW>
__device__ __forceinline__ void tile_body(const Args& a, int mat0, int c0, int64_t row_base, int rows, int m0,
                                          const uint32_t* my_pairs, uint8_t* smem) {
  constexpr int SB = s_bytes(KIND), DB = d_bytes(KIND);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, q = lane >> 4;
  const int KS = a.ks, nb = a.K >> 8;
  const int ks = wave & (KS - 1), cw = wave / KS;
  constexpr int GC = MODE == kGateUp ? CT / 2 : CT;  // column tiles of one matrix a wavefront has
  constexpr int LD = 16 * CT + kPad, HALVES = MODE == kGateUp ? 2 : 1, NB = chunks_held(ROWS);
  const int O = a.m[mat0].O, cols = (NW / KS) * GC * 16;  // the workgroup's columns of one matrix
  float* red = reinterpret_cast<float*>(smem);

  // the scales of the workgroup's rows: one run of bytes in each tensor of each half (what would
  // pass the matrix's end repeats its last 16 bytes: rows that are never stored)
  const int s_len = cols * nb * SB, d_len = cols * nb * DB;
  const uint8_t* code[2];
#pragma unroll
  for (int i = 0; i < HALVES; ++i) {
    const Mat& m = a.m[mat0 + i];
    code[i] = uniform(m.q + row_base * nb * q_bytes(KIND));
    const uint8_t *gs = uniform(m.s + (row_base + c0) * nb * SB), *gd = uniform(m.d + (row_base + c0) * nb * DB);
    const int s_end = (O - c0) * nb * SB - 16, d_end = (O - c0) * nb * DB - 16;
    const uint32_t at = lds_address(smem + x_bytes(ROWS, NW)) + i * (s_len + d_len);
    for (int p = wave * 1024; p < s_len; p += NW * 1024)
      if (p + 16 * lane < s_len) dma16(gs, (uint32_t)min(p + 16 * lane, s_end), at + p);
    for (int p = wave * 1024; p < d_len; p += NW * 1024)
      if (p + 16 * lane < d_len) dma16(gd, (uint32_t)min(p + 16 * lane, d_end), at + s_len + p);
  }
  if constexpr (HALVES == 1) code[1] = code[0];

  Work<KIND, RT, CT, NB> w;
  const int lr = cw * GC * 16 + c;  // of tile 0, which of the workgroup's rows
  w.ls0 = x_bytes(ROWS, NW) + (lr * nb + ks) * SB;
  w.ld0 = x_bytes(ROWS, NW) + s_len + (lr * nb + ks) * DB;
#pragma unroll
  for (int j = 0; j < CT; ++j) {
    w.ls_[j] = (j / GC) * (s_len + d_len) + (j % GC) * 16 * nb * SB;
    w.ld_[j] = (j / GC) * (s_len + d_len) + (j % GC) * 16 * nb * DB;
  }
  // this lane fetches a piece of rows 8 i + (lane >> 3)
  uint32_t xo[2 * RT];
#pragma unroll
  for (int i = 0; i < 2 * RT; ++i) {
    // rows past the end read a valid row: what they produce is never stored
    const int r = 8 * i + (lane >> 3);
    uint32_t src;
    if constexpr (MODE == kPlain) {
      src = (uint32_t)min(m0 + r, a.M - 1);
    } else {
      const uint32_t p = my_pairs[min(r, rows - 1)];
      src = a.up_div == 1 ? p : (int)p < a.pairs ? p / (uint32_t)a.up_div : p - (uint32_t)a.pairs;
    }
    xo[i] = 2 * src * (uint32_t)a.K;
  }
  const uint8_t* xs = smem + wave * (x_bytes(ROWS, NW) / NW);
  w.template run<GC>(code, c0 + lr, O, a.x, xo, nb, ks, KS, lane, smem, xs, lds_address(xs),
                     [&]() { __syncthreads(); });  // every wavefront's share of the scales has arrived
  __syncthreads();
  // The partial tiles meet in LDS. First the upper half of the K split hands its registers to
  // the lower half as they are (16 bytes a lane), which halves what the second pass holds.
  const int HS = KS / 2;
  {
    f32x4_t* raw = reinterpret_cast<f32x4_t*>(red) + (size_t)(cw * HS + (ks & (HS - 1))) * (RT * CT * 64) + lane;
    if (ks >= HS) {
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int j = 0; j < CT; ++j) raw[(r * CT + j) * 64] = w.acc[r][j];
    }
    __syncthreads();
    if (ks < HS) {
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int j = 0; j < CT; ++j) w.acc[r][j] += raw[(r * CT + j) * 64];
    }
    __syncthreads();
  }
  // D[row = 4 q + e][column = c]
  if (ks < HS) {
    float* mine = red + (cw * HS + ks) * (ROWS * LD);
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int j = 0; j < CT; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) mine[(16 * r + 4 * q + e) * LD + 16 * j + c] = w.acc[r][j][e];
  }
  __syncthreads();
  // four output columns a thread: the remaining partial sums in ks order
  const int quads = cols / 4;  // of a row
  const int n = rows * quads;
  for (int i = tid; i < n; i += 64 * NW) {
    const int row = i / quads, c4 = i - row * quads;
    const int w0 = (c4 / (4 * GC)) * HS, lc = 4 * (c4 % (4 * GC));
    const float* p = red + (w0 * ROWS + row) * LD + lc;
    f32x4_t v = *reinterpret_cast<const f32x4_t*>(p), u;
    for (int k = 1; k < HS; ++k) v += *reinterpret_cast<const f32x4_t*>(p + k * ROWS * LD);
    if constexpr (MODE == kGateUp) {
      u = *reinterpret_cast<const f32x4_t*>(p + 16 * GC);
      for (int k = 1; k < HS; ++k) u += *reinterpret_cast<const f32x4_t*>(p + 16 * GC + k * ROWS * LD);
    }
    const int col = c0 + 4 * c4;
    if (col >= O) continue;
    int64_t dst = m0 + row;
    if constexpr (MODE != kPlain) dst = my_pairs[row];
    bf16_t* y = a.m[mat0].y + dst * O + col;
    u32x2_t o;
    if constexpr (MODE == kGateUp) {
      o[0] = (uint32_t)swiglu_bf16(v[0], u[0]) | ((uint32_t)swiglu_bf16(v[1], u[1]) << 16);
      o[1] = (uint32_t)swiglu_bf16(v[2], u[2]) | ((uint32_t)swiglu_bf16(v[3], u[3]) << 16);
    } else {
      o[0] = dm_f2bf2(v[0], v[1]);
      o[1] = dm_f2bf2(v[2], v[3]);
    }
    if ((O & 3) == 0) {
      *reinterpret_cast<u32x2_t*>(y) = o;
    } else {  // (rows of y are not 8-byte aligned, and the last quad may be ragged)
      y[0] = (bf16_t)(o[0] & 0xffffu);
      if (col + 1 < O) y[1] = (bf16_t)(o[0] >> 16);
      if (col + 2 < O) y[2] = (bf16_t)(o[1] & 0xffffu);
      if (col + 3 < O) y[3] = (bf16_t)(o[1] >> 16);
    }
  }
}

// AFF: affine formats, else k-quants. NW wavefronts, grid (column blocks, row tiles), K >= 512.
template <bool AFF, int CT, int MODE, int ROWS, int NW>
__device__ __forceinline__ void body(const Args& a) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t nmm_smem[];
  constexpr int GC = MODE == kGateUp ? CT / 2 : CT;
  const int cols = (NW / a.ks) * GC * 16;
  int mat0 = 0, cb = blockIdx.x, rows, m0 = 0;
  int64_t row_base = 0;
  const uint32_t* my_pairs = nullptr;
  if constexpr (MODE == kPlain) {
#pragma unroll
    for (int i = 1; i < 4; ++i)
      if (i < a.n && (int)blockIdx.x >= a.m[i].cb0) {
        mat0 = i;
        cb = (int)blockIdx.x - a.m[i].cb0;
      }
    m0 = blockIdx.y * ROWS;
    rows = min(ROWS, a.M - m0);
  } else {
    const uint32_t tile = blockIdx.y;
    if (tile >= *a.n_tiles) return;
    const uint32_t e = __builtin_amdgcn_readfirstlane(a.tile_expert[tile]);
    rows = __builtin_amdgcn_readfirstlane((int)a.tile_count[tile]);
    my_pairs = a.pair + __builtin_amdgcn_readfirstlane(a.tile_start[tile]);
    if ((int)e >= a.E)
      mat0 = 2;
    else
      row_base = (int64_t)e * a.m[0].O;
  }
  const int c0 = cb * cols;
  const int kind = a.m[mat0].kind;
#define NMM_TILE(KIND, RT) tile_body<KIND, (RT <= ROWS / 16 ? RT : 1), CT, MODE, ROWS, NW>(a, mat0, c0, row_base, rows, m0, my_pairs, nmm_smem)
#define NMM_KIND(KIND)                                     \
  do {                                                     \
    if (rows <= 16 || ROWS == 16) NMM_TILE(KIND, 1);       \
    else if (rows <= 32 || ROWS <= 32) NMM_TILE(KIND, 2);  \
    else if (rows <= 48) NMM_TILE(KIND, 3);                \
    else NMM_TILE(KIND, 4);                                \
  } while (0)
  if constexpr (AFF) {
    if (kind == kA4) NMM_KIND(kA4);
    else NMM_KIND(kA8);
  } else {
    if (kind == kQ4K) NMM_KIND(kQ4K);
    else NMM_KIND(kQ6K);
  }
#undef NMM_KIND
#undef NMM_TILE
}

}  // namespace nmm
