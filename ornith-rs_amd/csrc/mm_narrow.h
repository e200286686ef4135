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
// The expert forms split columns, not K: an expert's tile takes thousands of workgroups whatever is split, and with K split
// a wavefront worked through two blocks only, with nothing in flight behind them, and spent a fifth of its vector
// instructions on partial sums. There a wavefront owns 32 columns over all of K (owned_tile()), its next block's codes in
// flight, and four wavefronts share the activations a block at a time. Many small workgroups beat fewer that do more
// (measured and not kept: eight wavefronts with K in halves, gate + up at 700 tokens 91 -> 123 us; four column groups a
// workgroup over resident activations, down 70 -> 74).
//
// What bounds the expert forms is vector issue beside the stream (700 tokens, gate + up: vector units 68 % of the time,
// matrix cores 15 %, 4.5 TB/s; with every expert's weights in L2 the launch still takes 80 of its 90 us). The codes' way to
// operands is 18 instructions for eight weights (scaled()). The plain launches of a short prompt are one pass of a
// chain: load, unpack, multiply, meet (vector units 13 %).
//
// Measured (us, before -> now): 12288 x 2048 Q4_K at 64 rows 29.5 -> 15.8 -> 14.8, 2048 x 4096 at 64 rows 52 -> 9.6 -> 7.2,
// 256 x 2048 Q6_K 28.6 -> 6.6 -> 5.4; the experts, gate + up + swiglu / down (the shared expert included): a 51-token prompt
// 104 / 49 -> 53 / 36 with K split -> 47 / 38 with columns owned, a 700-token one 156 / 76 -> 122 / 81 -> 90 / 69, over 4-bit
// affine weights at 600 tokens 109 / 62 -> 98 / 51; a 600-token prompt over 4-bit affine weights as a whole 461 ms
// (mat-vecs, row by row) -> 15.9 -> 13.2 ms.
//
// There are two orders of the sums, both by K alone: with K split over the wavefronts, 256-wide blocks, wavefront ks takes blocks ks,
// ks + KS, ... and the partial sums are added in one order; with columns owned (expert forms and kTall), all blocks in turn.
// Which one a plain matrix takes hangs on its own rows, columns and format (tall() in mm_narrow_kq.hip), never on the launch's
// other matrices or its tile.
//
// Weight formats:
//   Q4_K, Q6_K        dequantized with kquant::dequantize's arithmetic and rounded to bf16, as in
//                     kq_mm.hip
//   affine 4 / 8 bit  the codes are exact bf16 numbers and go to the matrix cores as they are; the
//                     sum over a group (32 / 64 k, one / two MFMAs) is multiplied by the group's
//                     scale in fp32, and the bias meets the group's sum of activations, which the
//                     matrix core makes from ones, four groups at a time in an fp32 product. No weight
//                     is rounded: the arithmetic is that of the mat-vec (linear.hip), summed in another order.
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
enum Mode { kPlain = 0, kGather = 1, kGateUp = 2, kTall = 3 };

struct Mat {
  const uint8_t* q;  // codes
  const uint8_t* s;  // k-quant scales; affine scales (bf16)
  const uint8_t* d;  // k-quant d (and dmin); affine biases (bf16)
  bf16_t* y;
  int O, kind;
  int cb0;  // plain form: first column block of the launch that is this matrix's
};

// Dense bf16 matrices that ride along with a plain launch: 16 x 16 tiles, numbered row tile by row tile, the matrices' column
// tiles laid end to end.
struct Riders {
  const bf16_t* w[2];
  bf16_t* y[2];
  int O[2];
  int tiles, wgs;  // column tiles; workgroups
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
  uint32_t up_magic;  // dm_div_magic(up_div)
  int tiles_max, blocks;  // room in the tile list; column blocks a tile
  Riders d;
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

// a barrier that leaves loads in flight
__device__ __forceinline__ void barrier_only() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
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
// s * h + o with h the lower (HI = 0) or upper 16 bits of w as an f16 number: one instruction, one rounding
template <int HI>
__device__ __forceinline__ float fma_half(float s, uint32_t w, float o) {
  float r;
  if constexpr (HI)
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[0,1,0] op_sel_hi:[0,1,0]" : "=v"(r) : "v"(s), "v"(w), "v"(o));
  else
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[0,0,0] op_sel_hi:[0,1,0]" : "=v"(r) : "v"(s), "v"(w), "v"(o));
  return r;
}
// w >> N (N < 0: w << -N). TAG makes it another instruction in every step that wants it: merged into one, the shifted words of a
// block would be kept from step to step (a hundred registers spilled).
template <int N, int TAG>
__device__ __forceinline__ uint32_t shifted(uint32_t w) {
  uint32_t r;
  if constexpr (N >= 0)
    asm("v_lshrrev_b32 %0, %1, %2 ; %3" : "=v"(r) : "n"(N), "v"(w), "n"(TAG));
  else
    asm("v_lshlrev_b32 %0, %1, %2 ; %3" : "=v"(r) : "n"(-N), "v"(w), "n"(TAG));
  return r;
}
// w = s * code + o of eight codes, rounded to bf16. A code of up to ten bits at the bottom of a half is, read as a
// (subnormal) f16 number, code * 2^-24, and four bits up code * 2^-20: no conversion, two codes a mask. s comes
// multiplied by the 2^24 or 2^20, which loses nothing, so the fma's product is the code's times the scale's, bit for bit.
// e0 / e1: codes 0, 2 and 4, 6; o0 / o1: codes 1, 3 and 5, 7.
__device__ __forceinline__ bf16x8_t scaled(uint32_t e0, uint32_t o0, uint32_t e1, uint32_t o1, float s, float o) {
  return as_frag(dm_f2bf2(fma_half<0>(s, e0, o), fma_half<0>(s, o0, o)), dm_f2bf2(fma_half<1>(s, e0, o), fma_half<1>(s, o0, o)),
                 dm_f2bf2(fma_half<0>(s, e1, o), fma_half<0>(s, o1, o)), dm_f2bf2(fma_half<1>(s, e1, o), fma_half<1>(s, o1, o)));
}

// Q4_K: lane q takes pieces q (steps 0 - 3) and q + 4 of the block's eight 16-byte code pieces; piece
// p is bytes 16 (p & 1) .. of 64-group p >> 1, low nibbles k = 64 (p >> 1) + 16 (p & 1) + i, high
// ones 32 further on. Chunk u = (half, nibble).
template <>
struct Tile<kQ4K> {
  static constexpr bool kAffine = false;
  static constexpr int kSteps = 1, kLoads = 2;
  struct Codes {
    u32x4_t w[2];
    __device__ __forceinline__ void here() { asm volatile("" : "+v"(w[0]), "+v"(w[1])); }
  } t;
  float dd, nm;     // d * 2^24, -dmin
  uint32_t sm;      // scales (low bytes) and minima of the half's two sub-blocks of this lane
  float s, o;
  static __device__ __forceinline__ int piece(int u, int slot) {
    return 16 * (u >> 1) + 4 * (u & 1) + 8 * (slot >> 2) + (slot & 3);
  }
  static constexpr int half_bytes() { return 256; }  // from chunk u's pieces to chunk u + 2's
  template <int H>
  static __device__ __forceinline__ int slot(int q) { return 2 * q + H; }
  static __device__ __forceinline__ void load(Codes& t, const uint8_t* cq, uint32_t blk, int q) {
    t.w[0] = ld_off<u32x4_t>(cq, blk * q_bytes(kQ4K) + 16 * q);
    t.w[1] = ld_off<u32x4_t>(cq + 64, blk * q_bytes(kQ4K) + 16 * q);
  }
  // sub-block 4 (u >> 1) + 2 (q >> 1) + (u & 1) of the block whose scales are at ls / ld in LDS
  template <int U>
  __device__ __forceinline__ void scales(const uint8_t* ls, const uint8_t* ld, int q) {
    const uint32_t* sc = reinterpret_cast<const uint32_t*>(ls);
    const uint32_t pick = q >> 1 ? 0x07060302u : 0x05040100u;
    if constexpr (U == 0) {
      const uint32_t dmw = *reinterpret_cast<const uint32_t*>(ld);
      dd = dm_h2f((f16_t)(dmw & 0xffffu)) * 16777216.f;
      nm = -dm_h2f((f16_t)(dmw >> 16));
      sm = __builtin_amdgcn_perm(sc[1], sc[0], pick) & 0x3f3f3f3fu;
    }
    if constexpr (U == 2)
      sm = __builtin_amdgcn_perm((sc[2] >> 4) & 0x0f0f0f0fu, sc[2] & 0x0f0f0f0fu, pick) |
           ((__builtin_amdgcn_perm(sc[1], sc[0], pick) >> 2) & 0x30303030u);
    // (the odd chunks hold the high nibbles, whose codes lie four bits up)
    s = ((U & 1) ? dd * 0.0625f : dd) * dm_ubyte<(U & 1)>(sm);
    o = nm * dm_ubyte<2 + (U & 1)>(sm);
  }
  template <int S>
  __device__ __forceinline__ bf16x8_t frag() const {
    constexpr uint32_t M = ((S >> 1) & 1) ? 0x00f000f0u : 0x000f000fu;
    const uint32_t a = t.w[S >> 2][2 * (S & 1)], b = t.w[S >> 2][2 * (S & 1) + 1];
    return scaled(a & M, shifted<8, S>(a) & M, b & M, shifted<8, S>(b) & M, s, o);
  }
};

// Q6_K: lane q takes positions 16 (q & 1) .. of the 128-half q >> 1: 16 bytes of each of the half's
// two low-nibble rows and of its high bits. Chunk u = quarter of the halves (k = 128 half + 32 u + position).
template <>
struct Tile<kQ6K> {
  static constexpr bool kAffine = false;
  static constexpr int kSteps = 1, kLoads = 3;
  struct Codes {
    u32x4_t la, lb, h;
    __device__ __forceinline__ void here() { asm volatile("" : "+v"(la), "+v"(lb), "+v"(h)); }
  } t;
  float s, o;
  static __device__ __forceinline__ int piece(int u, int slot) { return 16 * (slot >> 2) + 4 * u + (slot & 3); }
  static constexpr int half_bytes() { return 128; }
  template <int H>
  static __device__ __forceinline__ int slot(int q) { return 2 * q + H; }
  static __device__ __forceinline__ void load(Codes& t, const uint8_t* cq, uint32_t blk, int q) {
    const uint32_t at = blk * q_bytes(kQ6K) + 64 * (q >> 1) + 16 * (q & 1);
    t.la = ld_off<u32x4_t>(cq, at);
    t.lb = ld_off<u32x4_t>(cq + 32, at);
    t.h = ld_off<u32x4_t>(cq + 128, blk * q_bytes(kQ6K) + 16 * q);
  }
  // scale 8 (q >> 1) + 2 u + (q & 1) of the block's sixteen
  template <int U>
  __device__ __forceinline__ void scales(const uint8_t* ls, const uint8_t* ld, int q) {
    const int8_t sc = (int8_t)ls[8 * (q >> 1) + 2 * U + (q & 1)];
    const float v = dm_h2f(*reinterpret_cast<const f16_t*>(ld)) * (float)(int)sc;
    s = v * (U < 2 ? 16777216.f : 1048576.f);
    o = -32.f * v;
  }
  // quarters 0 and 1 are low nibbles (the codes lie at the bottom of their halves), 2 and 3 high ones (four bits up)
  template <int S>
  __device__ __forceinline__ bf16x8_t frag() const {
    constexpr int QD = S >> 1, NIB = QD >> 1, W = 2 * (S & 1), SH = 4 - 2 * (QD & 1);
    constexpr uint32_t M = NIB ? 0x00f000f0u : 0x000f000fu, MH = NIB ? 0x03000300u : 0x00300030u;
    const u32x4_t& lo = (QD & 1) ? t.lb : t.la;
    const uint32_t a = lo[W], b = lo[W + 1], ha = t.h[W], hb = t.h[W + 1];
    return scaled((a & M) | (shifted<-SH, S>(ha) & MH), (shifted<8, S>(a) & M) | (shifted<8 - SH, S>(ha) & MH), (b & M) | (shifted<-SH, S>(hb) & MH),
                  (shifted<8, S>(b) & M) | (shifted<8 - SH, S>(hb) & MH), s, o);
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
  static constexpr int kSteps = 1, kLoads = 2;  // k steps a group
  struct Codes {
    u32x4_t t[2];  // word q of groups 4 i + g
    __device__ __forceinline__ void here() { asm volatile("" : "+v"(t[0]), "+v"(t[1])); }
  } t;
  u32x4_t sc;  // the block's eight scales, two to a word
  static __device__ __forceinline__ int piece(int u, int slot) { return 8 * u + slot; }
  static constexpr int half_bytes() { return 256; }
  template <int H>
  static __device__ __forceinline__ int slot(int q) { return 4 * H + q; }
  static __device__ __forceinline__ void load(Codes& t, const uint8_t* cq, uint32_t blk, int q) {
    // whole groups (16 bytes): lane q holds group 4 i + q
    t.t[0] = ld_off<u32x4_t>(cq, blk * q_bytes(kA4) + 16 * q);
    t.t[1] = ld_off<u32x4_t>(cq + 64, blk * q_bytes(kA4) + 16 * q);
  }
  // word g of group q -> word q of group g: the 4 x 4 transpose over the lanes of a column
  template <int I>
  __device__ __forceinline__ void transpose() {
    uint32_t a = t.t[I][0], b = t.t[I][1], c = t.t[I][2], d = t.t[I][3];
    swap_rows<32>(a, c);
    swap_rows<32>(b, d);
    swap_rows<16>(a, b);
    swap_rows<16>(c, d);
    t.t[I] = u32x4_t{a, b, c, d};
  }
  template <int U>
  __device__ __forceinline__ void scales(const uint8_t* ls, const uint8_t*, int) {
    if constexpr (U == 0) {
      transpose<0>();
      sc = *reinterpret_cast<const u32x4_t*>(ls);
    }
    if constexpr (U == 2) transpose<1>();
  }
  template <int S>
  __device__ __forceinline__ float scale() const { return (S & 1) ? dm_bf2f_hi(sc[S >> 1]) : dm_bf2f_lo(sc[S >> 1]); }
  template <int S>
  __device__ __forceinline__ bf16x8_t frag() const {
    const uint32_t w = t.t[S >> 2][S & 3];
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
  static constexpr int kSteps = 2, kLoads = 8;
  struct Codes {
    u32x2_t w[8];
    __device__ __forceinline__ void here() {
      asm volatile("" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3]), "+v"(w[4]), "+v"(w[5]), "+v"(w[6]), "+v"(w[7]));
    }
  } t;
  u32x2_t sc;  // the block's four scales
  static __device__ __forceinline__ int piece(int u, int slot) { return 8 * u + slot; }
  static constexpr int half_bytes() { return 256; }
  template <int H>
  static __device__ __forceinline__ int slot(int q) { return 4 * H + q; }
  static __device__ __forceinline__ void load(Codes& t, const uint8_t* cq, uint32_t blk, int q) {
#pragma unroll
    for (int i = 0; i < 8; ++i) t.w[i] = ld_off<u32x2_t>(cq + 32 * i, blk * q_bytes(kA8) + 8 * q);
  }
  template <int U>
  __device__ __forceinline__ void scales(const uint8_t* ls, const uint8_t*, int) {
    if constexpr (U == 0) sc = *reinterpret_cast<const u32x2_t*>(ls);
  }
  template <int S>
  __device__ __forceinline__ float scale() const { return (S & 2) ? dm_bf2f_hi(sc[S >> 2]) : dm_bf2f_lo(sc[S >> 2]); }
  template <int S>
  __device__ __forceinline__ bf16x8_t frag() const {  // 0 .. 255 are bf16 numbers
    const uint32_t a = t.w[S][0], b = t.w[S][1];
    return as_frag(dm_f2bf2(dm_ubyte<0>(a), dm_ubyte<1>(a)), dm_f2bf2(dm_ubyte<2>(a), dm_ubyte<3>(a)),
                   dm_f2bf2(dm_ubyte<0>(b), dm_ubyte<1>(b)), dm_f2bf2(dm_ubyte<2>(b), dm_ubyte<3>(b)));
  }
};

// ---- one wavefront's share: RT x CT tiles of 16 x 16 over its K blocks ----------------------------
// NB: activation chunks (2 KB * RT each) its part of LDS holds
// PF: the codes of the wavefront's next block are asked for while it works on this one (plain form)
template <int KIND, int RT, int CT, int NB, bool PF>
struct Work {
  typedef Tile<KIND> T;
  f32x4_t acc[RT][CT];
  T t[CT];
  float sx[RT];           // affine: the row's sum over group (its lane quarter) of the last four groups
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
      constexpr int N = T::kSteps, G = S / N;  // group of the block
      const bf16x8_t ones = as_frag(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u);
      const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
      bf16x8_t a1[RT];
      read(std::integral_constant<int, H>{}, a);
      if constexpr (N == 2) read(std::integral_constant<int, 1>{}, a1);
      // the rows' sums over the group: ones times the activations' transpose puts row c's into lane c of every
      // quarter, and quarter q keeps group q's, which is the operand layout of the fp32 product below
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        f32x4_t v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, a[r], zero, 0, 0, 0);
        if constexpr (N == 2) v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, a1[r], v, 0, 0, 0);
        sx[r] = q == (G & 3) ? v[0] : sx[r];
        // (v's other elements stay taken until its product has ended: their registers would go to the unpacking's inline
        // assembly at once, which the compiler does not hold back for a matrix instruction in flight)
        asm volatile("" : "+v"(sx[r]) : "v"(v));
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
          for (int e = 0; e < 4; ++e) acc[r][j][e] = dm_fma(t[j].template scale<S>(), g[r][e], acc[r][j][e]);
      }
      // the biases of four groups against the rows' sums over them, fp32 on the matrix cores (an fma an
      // element and group beside the scale's was a third of the vector work)
      if constexpr ((G & 3) == 3) {
#pragma unroll
        for (int j = 0; j < CT; ++j) {
          const float bias = dm_bf2f(*reinterpret_cast<const bf16_t*>(smem + ld0 + ld_[j] + 2 * ((G & 4) + q)));
#pragma unroll
          for (int r = 0; r < RT; ++r) acc[r][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(sx[r], bias, acc[r][j], 0, 0, 0);
        }
      }
    }
    // (or the scheduler dequantizes the whole block ahead, and spills)
    __builtin_amdgcn_sched_barrier(0);
  }
  // codes of block ib of weight row `row` of O
  static __device__ __forceinline__ void load(typename T::Codes& d, const uint8_t* code, int row, int O, int ib, int nb, int q) {
    T::load(d, code + (size_t)ib * q_bytes(KIND), (uint32_t)min(row, O - 1) * (uint32_t)nb, q);
  }
  // the first block's codes, ahead of what the activations' addresses wait for. code: of the two matrices (GC column
  // tiles each); row0: the lane's weight row of tile 0
  template <int GC>
  __device__ __forceinline__ void start(const uint8_t* const (&code)[CT / GC], int row0, int O, int nb, int ks, int lane) {
#pragma unroll
    for (int j = 0; j < CT; ++j) load(t[j].t, code[j / GC], row0 + 16 * (j % GC), O, ks, nb, lane >> 4);
    __builtin_amdgcn_sched_barrier(0);
  }
  static constexpr int kScaleLoads = KIND == kA4 ? 2 : 0;
  // The plain form: one block, with two chunks and the codes of it asked for. MORE: the wavefront has another one, KS blocks
  // on; its codes go out here behind this block's activations (which are waited for one by one), its activations as
  // this block's buffers come free.
  template <bool MORE, class F, class G>
  __device__ __forceinline__ void block(const uint8_t* code, int row0, int O, const uint8_t* xk, const uint32_t (&xo)[2 * RT], int ib,
                                        int nb, int KS, int lane, const uint8_t* smem, const uint8_t* xs, uint32_t lds, F first, G scales) {
    static_assert(NB == 2, "two chunks in flight");
    const int c = lane & 15, q = lane >> 4;
    constexpr bool AHEAD = MORE && PF;
    constexpr int NL = (AHEAD ? CT * T::kLoads : 0) + (MORE ? kScaleLoads : 0);
    const uint8_t* const xn = xk + (size_t)KS * 512;
    typename T::Codes next[CT];
    wait_loads<0>();
    first();
    step<0>(smem, xs, c, q);
    step<1>(smem, xs, c, q);
    fetch<2>(xk, xo, lds, lane);
    step<2>(smem, xs, c, q);
    step<3>(smem, xs, c, q);
    fetch<3>(xk, xo, lds, lane);
    if constexpr (AHEAD) {
#pragma unroll
      for (int j = 0; j < CT; ++j) load(next[j], code, row0 + 16 * j, O, ib + KS, nb, q);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (MORE) scales(ib + KS);
    wait_loads<2 * RT + NL>();
    step<4>(smem, xs, c, q);
    step<5>(smem, xs, c, q);
    if constexpr (MORE) fetch<0>(xn, xo, lds, lane);
    wait_loads<NL + (MORE ? 2 * RT : 0)>();
    step<6>(smem, xs, c, q);
    step<7>(smem, xs, c, q);
    if constexpr (MORE) {
      fetch<1>(xn, xo, lds, lane);
#pragma unroll
      for (int j = 0; j < CT; ++j) {
        if constexpr (PF) t[j].t = next[j];
        else load(t[j].t, code, row0 + 16 * j, O, ib + KS, nb, q);
      }
    }
  }
  // The form whose wavefronts own columns: every one works through all of K, a block at a time, and the workgroup's four
  // share the block's activations, chunk U at xs + U * RT * 2 KB. They come in two chunks a piece (wavefront `wave` fetches
  // half the rows of chunk `wave & 1` of a half block: xo, lds) or whole blocks (chunk `wave`):
  //   whole blocks in two buffers, each asked for a block ahead;
  //   HALF: half blocks in the halves of one buffer, each asked for half a block ahead.
  // MORE: the next block's activations and codes go out here.
  __device__ __forceinline__ static void ask_block(const uint8_t* x, const uint32_t (&xo)[2 * RT], uint32_t lds) {
#pragma unroll
    for (int i = 0; i < 2 * RT; ++i) dma16(x, xo[i], lds + i * 1024);
  }
  __device__ __forceinline__ static void ask_half(const uint8_t* x, const uint32_t (&xo)[2 * RT], int half, uint32_t lds) {
#pragma unroll
    for (int i = 0; i < RT; ++i) dma16(x + half * T::half_bytes(), xo[i], lds + half * (RT * 4096) + i * 1024);
  }
  template <int GC, bool HALF, bool FIRST, bool MORE, class F>
  __device__ __forceinline__ void owned_block(const uint8_t* const (&code)[CT / GC], int row0, int O, const uint8_t* x,
                                              const uint32_t (&xo)[2 * RT], int ib, int nb, int lane, const uint8_t* smem,
                                              const uint8_t* xs, uint32_t lds, F ask_scales) {
    const int c = lane & 15, q = lane >> 4;
    typename T::Codes next[CT];
    auto ask_codes = [&]() {
#pragma unroll
      for (int j = 0; j < CT; ++j) load(next[j], code[j / GC], row0 + 16 * (j % GC), O, ib + 1, nb, q);
      __builtin_amdgcn_sched_barrier(0);
    };
    const int buf = HALF ? 0 : (ib & 1) * (RT * 8192);
    // this block's activations (their first half) were asked for ahead of its codes
    wait_loads<FIRST ? 0 : CT * T::kLoads>();
    barrier_only();
    if constexpr (HALF) {
      // (This block's codes are used next: waited for here, since behind the request that follows the compiler waits for that as
      // well, half a block early. 4-bit affine, us: gate + up at 600 tokens 96.8 / 94.0, 12288 x 2048 at 512 / 2000 rows 59 / 57 and
      // 194 / 190; Q4_K level.)
#pragma unroll
      for (int j = 0; j < CT; ++j) t[j].t.here();
      ask_half(x, xo, 1, lds);
    } else if constexpr (MORE) {
      ask_block(x + 512, xo, lds + ((ib + 1) & 1) * (RT * 8192));
      ask_scales(ib + 1);
      ask_codes();
    }
    step<0>(smem, xs + buf, c, q);
    step<1>(smem, xs + buf, c, q);
    step<2>(smem, xs + buf, c, q);
    step<3>(smem, xs + buf, c, q);
    if constexpr (HALF) {
      wait_loads<0>();
      barrier_only();
      if constexpr (MORE) {
        ask_half(x + 512, xo, 0, lds);
        ask_scales(ib + 1);
        ask_codes();
      }
    }
    step<4>(smem, xs + buf, c, q);
    step<5>(smem, xs + buf, c, q);
    step<6>(smem, xs + buf, c, q);
    step<7>(smem, xs + buf, c, q);
    if constexpr (MORE) {
#pragma unroll
      for (int j = 0; j < CT; ++j) t[j].t = next[j];
    }
  }
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      sx[r] = 0.f;
#pragma unroll
      for (int j = 0; j < CT; ++j) acc[r][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
  }
  // x, xo: the activations and the byte offsets of the rows this lane fetches; xs / lds: this wavefront's
  // activation buffers; scales_here(): what has to be done before the first block's arithmetic. start() has been called.
  // scales(ib) as above, scales_of(ib): ls0 and ld0 of a block.
  template <class F, class G, class S>
  __device__ __forceinline__ void run(const uint8_t* code, int row0, int O, const bf16_t* x, const uint32_t (&xo)[2 * RT], int nb, int ks,
                                      int KS, int lane, const uint8_t* smem, const uint8_t* xs, uint32_t lds, F scales_here, G scales,
                                      S scales_of) {
    clear();
    const uint8_t* xk = reinterpret_cast<const uint8_t*>(x) + (size_t)ks * 512;
    fetch<0>(xk, xo, lds, lane);
    fetch<1>(xk, xo, lds, lane);
    int ib = ks;
    auto first = [&]() {
      if (ib == ks) scales_here();
    };
    for (; ib + KS < nb; ib += KS, xk += (size_t)KS * 512) {
      scales_of(ib);
      block<true>(code, row0, O, xk, xo, ib, nb, KS, lane, smem, xs, lds, first, scales);
    }
    scales_of(ib);
    block<false>(code, row0, O, xk, xo, ib, nb, KS, lane, smem, xs, lds, first, scales);
  }
};

constexpr int kLdsBytes = 160 * 1024;
constexpr int kPad = 4;  // a row of a partial tile: 16 CT + 4 floats, so the four 4-row groups of a store hit other banks

// LDS of a workgroup: activation chunks of its NW wavefronts, then the scales of its rows; the
// partial tiles go over both (host and device share the arithmetic)
__host__ __device__ constexpr int x_bytes(int rows, int nw) { return nw * 2 * (rows / 16) * 2048; }
__host__ __device__ constexpr int red_bytes(int rows, int ct, int nw) { return nw / 2 * rows * (16 * ct + kPad) * 4; }

// the plain form: a workgroup's tile of up to 16 RT rows (of ROWS): partial products, their sums, the outputs
template <int KIND, int RT, int CT, int ROWS, int NW>
__device__ __forceinline__ void tile_body(const Args& a, int mat, int c0, int rows, int m0, uint8_t* smem) {
  constexpr int SB = s_bytes(KIND), DB = d_bytes(KIND);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, q = lane >> 4;
  const int KS = a.ks, nb = a.K >> 8;
  const int ks = wave & (KS - 1), cw = wave / KS;
  constexpr int LD = 16 * CT + kPad;
  const Mat& m = a.m[mat];
  const int O = m.O, cols = (NW / KS) * CT * 16;  // the workgroup's columns
  float* red = reinterpret_cast<float*>(smem);

  // The scales: of the workgroup's rows over all of K, one run of bytes in each tensor (what would pass the matrix's end
  // repeats its last 16 bytes: rows that are never stored). 4-bit affine, whose 16-byte pieces can be fetched one
  // by one: of the wavefront's columns, a block ahead in two buffers (all of K = 4096 would be 32 KB and leave a compute
  // unit one workgroup: 2048 x 4096 at 600 rows 48 us).
  constexpr bool RING = KIND == kA4;
  const int s_len = cols * nb * SB, d_len = cols * nb * DB;
  const uint8_t* const code[1] = {uniform(m.q)};
  const int lr = cw * CT * 16 + c;  // of tile 0, which of the workgroup's rows
  const uint8_t *gs = uniform(m.s + (int64_t)c0 * nb * SB), *gd = uniform(m.d + (int64_t)c0 * nb * DB);
  const uint32_t ring = x_bytes(ROWS, NW) + wave * 4096;
  const uint32_t ring_at = lds_address(smem + ring), ring_off = (uint32_t)min(cw * CT * 16 + lane, O - c0 - 1) * (uint32_t)(nb * 16);
  auto ask_scales = [&](int ib) {
    if constexpr (RING) {
      dma16(gs + ib * 16, ring_off, ring_at + (ib / KS & 1) * 2048);
      dma16(gd + ib * 16, ring_off, ring_at + (ib / KS & 1) * 2048 + 1024);
    }
  };
  if constexpr (!RING) {
    const int s_end = (O - c0) * nb * SB - 16, d_end = (O - c0) * nb * DB - 16;
    const uint32_t at = lds_address(smem + x_bytes(ROWS, NW));
    for (int p = wave * 1024; p < s_len; p += NW * 1024)
      if (p + 16 * lane < s_len) dma16(gs, (uint32_t)min(p + 16 * lane, s_end), at + p);
    for (int p = wave * 1024; p < d_len; p += NW * 1024)
      if (p + 16 * lane < d_len) dma16(gd, (uint32_t)min(p + 16 * lane, d_end), at + s_len + p);
  }
  ask_scales(ks);

  // (the codes ahead where the registers hold two blocks of them)
  Work<KIND, RT, CT, 2, (KIND == kQ4K || KIND == kA4) && RT <= 2> w;
  w.template start<CT>(code, c0 + lr, O, nb, ks, lane);
  auto scales_of = [&](int ib) {
    w.ls0 = RING ? ring + (ib / KS & 1) * 2048 + c * 16 : x_bytes(ROWS, NW) + (lr * nb + ib) * SB;
    w.ld0 = RING ? w.ls0 + 1024 : x_bytes(ROWS, NW) + s_len + (lr * nb + ib) * DB;
  };
#pragma unroll
  for (int j = 0; j < CT; ++j) {
    w.ls_[j] = RING ? j * 256 : j * 16 * nb * SB;
    w.ld_[j] = RING ? j * 256 : j * 16 * nb * DB;
  }
  // this lane fetches a piece of rows 8 i + (lane >> 3); rows past the end read a valid row: what they produce is never stored
  uint32_t xo[2 * RT];
#pragma unroll
  for (int i = 0; i < 2 * RT; ++i) xo[i] = 2 * (uint32_t)min(m0 + 8 * i + (lane >> 3), a.M - 1) * (uint32_t)a.K;
  const uint8_t* xs = smem + wave * (x_bytes(ROWS, NW) / NW);
  w.run(code[0], c0 + lr, O, a.x, xo, nb, ks, KS, lane, smem, xs, lds_address(xs),
        [&]() { barrier_only(); },  // every wavefront's share of the scales has arrived (waited for by each)
        ask_scales, scales_of);
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
    const int w0 = (c4 / (4 * CT)) * HS, lc = 4 * (c4 % (4 * CT));
    const float* p = red + (w0 * ROWS + row) * LD + lc;
    f32x4_t v = *reinterpret_cast<const f32x4_t*>(p);
    for (int k = 1; k < HS; ++k) v += *reinterpret_cast<const f32x4_t*>(p + k * ROWS * LD);
    const int col = c0 + 4 * c4;
    if (col >= O) continue;
    bf16_t* y = m.y + (int64_t)(m0 + row) * O + col;
    const u32x2_t o = {dm_f2bf2(v[0], v[1]), dm_f2bf2(v[2], v[3])};
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

// The forms whose wavefronts own columns: an expert's tile, or (kTall) 64 rows of a plain product, takes four wavefronts a block
// of 128 columns (64 of gate and of up); each owns 32 of them over all of K, its codes a block ahead in registers, so
// nothing has to meet at the end.
// LDS: activations, and the scales of 128 rows over all of K (4-bit affine: 32 KB at K = 2048, 16 KB the others). What
// makes room for another workgroup a compute unit where those two are too much: HALF, the activations half a block at a time
// (64-row tiles; 4-bit affine gate + up, 106 -> 98 us at 600 tokens; elsewhere the second barrier a block costs more), and RING,
// the scales of two blocks (4-bit affine, 64-row tiles, 71 -> 61 us at 12288 x 2048 and 600 rows; it is 64 lookups a load, which
// an expert's gate + up has no room for: 59 -> 73 us at 40 tokens).
__host__ __device__ constexpr bool owned_half(int kind, int mode) { return mode == kTall || (kind == kA4 && mode == kGateUp); }
__host__ __device__ constexpr bool owned_ring(int kind, int mode) { return mode == kTall && kind == kA4; }
__host__ __device__ constexpr int owned_x_bytes(int rows, int kind, int mode) { return rows * (owned_half(kind, mode) ? 512 : 1024); }
__host__ __device__ constexpr int owned_lds(int rows, int kind, int mode, int nb) {
  return owned_x_bytes(rows, kind, mode) + 128 * (owned_ring(kind, mode) ? 2 : nb) * (s_bytes(kind) + d_bytes(kind));
}
template <int KIND, int RT, int MODE>
__device__ __forceinline__ void owned_tile(const Args& a, int mat0, int c0, int64_t row_base, int rows, int m0, const uint32_t* my_pairs,
                                           uint8_t* smem) {
  constexpr int SB = s_bytes(KIND), DB = d_bytes(KIND), CT = 2, HALVES = MODE == kGateUp ? 2 : 1, GC = CT / HALVES;
  constexpr bool HALF = owned_half(KIND, MODE), RING = owned_ring(KIND, MODE);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, q = lane >> 4;
  const int nb = a.K >> 8, O = a.m[mat0].O;
  constexpr int cols = 4 * GC * 16;  // the workgroup's columns of one matrix
  typedef Work<KIND, RT, CT, 4, true> W;
  // The activations' addresses take a trip to memory of their own (the pairs), the weights are the longest one:
  // the pairs go out first, the scales and the first codes behind them, and the activations when the pairs are here.
  uint32_t pr[2 * RT];
  constexpr int NP = HALF ? RT : 2 * RT;
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int r = min(8 * ((HALF ? RT * (wave >> 1) : 0) + i) + (lane >> 3), rows - 1);
    if constexpr (MODE == kTall) pr[i] = m0 + r;
    else pr[i] = my_pairs[r];
  }
  __builtin_amdgcn_sched_barrier(0);
  const int s_len = RING ? cols * 16 : cols * nb * SB, d_len = cols * nb * DB, s_at = owned_x_bytes(16 * RT, KIND, MODE);
  // 4-bit affine over all of K: a row's blocks (16 bytes of scales, 16 of biases each) lie at block ^ (row & 7), or the
  // sixteen rows of a tile would be read from two places of the banks
  const bool turned = KIND == kA4 && !RING && nb % 8 == 0;
  auto from = [&](int p) { return turned ? p ^ (((p / (16 * nb)) & 7) << 4) : p; };
  const uint8_t* code[HALVES];
#pragma unroll
  for (int i = 0; i < HALVES; ++i) {
    const Mat& m = a.m[mat0 + i];
    code[i] = uniform(m.q + row_base * nb * q_bytes(KIND));
    if constexpr (!RING) {
      const uint8_t *gs = uniform(m.s + (row_base + c0) * nb * SB), *gd = uniform(m.d + (row_base + c0) * nb * DB);
      const int s_end = (O - c0) * nb * SB - 16, d_end = (O - c0) * nb * DB - 16;
      const uint32_t at = lds_address(smem + s_at) + i * (s_len + d_len);
      for (int p = wave * 1024; p < s_len; p += 4096)
        if (p + 16 * lane < s_len) dma16(gs, (uint32_t)min(from(p + 16 * lane), s_end), at + p);
      for (int p = wave * 1024; p < d_len; p += 4096)
        if (p + 16 * lane < d_len) dma16(gd, (uint32_t)min(from(p + 16 * lane), d_end), at + s_len + p);
    }
  }
  // RING: wavefronts 0, 1 fetch the scales of 64 rows each (of a matrix each), 2, 3 the biases
  const uint8_t* ring_from = nullptr;
  uint32_t ring_off = 0;
  const uint32_t ring_at = lds_address(smem + s_at) + wave * 1024;
  if constexpr (RING) {
    const Mat& m = a.m[mat0 + (HALVES == 2 ? wave & 1 : 0)];
    ring_from = uniform((wave >> 1 ? m.d : m.s) + (row_base + c0) * nb * 16);
    ring_off = (uint32_t)min((HALVES == 2 ? 0 : 64 * (wave & 1)) + lane, O - c0 - 1) * (uint32_t)(nb * 16);
  }
  auto ask_scales = [&](int ib) {
    if constexpr (RING) dma16(ring_from + ib * 16, ring_off, ring_at + (ib & 1) * 4096);
  };
  ask_scales(0);
  W w;
  const int lr = wave * GC * 16 + c;
  w.template start<GC>(code, c0 + lr, O, nb, 0, lane);
#pragma unroll
  for (int j = 0; j < CT; ++j) {
    w.ls_[j] = RING ? (j / GC) * s_len + (j % GC) * 256 : (j / GC) * (s_len + d_len) + (j % GC) * 16 * nb * SB;
    w.ld_[j] = RING ? (j / GC) * s_len + (j % GC) * 256 : (j / GC) * (s_len + d_len) + (j % GC) * 16 * nb * DB;
  }
  w.clear();
  uint32_t xo[2 * RT];
  const uint32_t piece = 16 * (uint32_t)Tile<KIND>::piece(HALF ? wave & 1 : wave, (lane & 7) ^ (lane >> 3));
  const uint32_t lds = lds_address(smem) + (HALF ? (wave & 1) * (RT * 2048) + (wave >> 1) * (RT * 1024) : wave * (RT * 2048));
  const uint8_t* x = reinterpret_cast<const uint8_t*>(a.x);
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const uint32_t p = pr[i], src = MODE == kTall || a.up_div == 1 ? p : (int)p < a.pairs ? dm_div(p, (uint32_t)a.up_div, a.up_magic) : p - (uint32_t)a.pairs;
    xo[i] = 2 * src * (uint32_t)a.K + piece;
  }
  if constexpr (HALF) W::ask_half(x, xo, 0, lds);
  else W::ask_block(x, xo, lds);
  auto scales_of = [&](int ib) {
    const int at = turned ? ib ^ (c & 7) : ib;
    w.ls0 = RING ? s_at + (ib & 1) * 4096 + lr * 16 : s_at + (lr * nb + at) * SB;
    w.ld0 = RING ? w.ls0 + 2048 : s_at + s_len + (lr * nb + at) * DB;
  };
  scales_of(0);
  w.template owned_block<GC, HALF, true, true>(code, c0 + lr, O, x, xo, 0, nb, lane, smem, smem, lds, ask_scales);
  for (int ib = 1; ib + 1 < nb; ++ib) {
    x += 512;
    scales_of(ib);
    w.template owned_block<GC, HALF, false, true>(code, c0 + lr, O, x, xo, ib, nb, lane, smem, smem, lds, ask_scales);
  }
  x += 512;
  scales_of(nb - 1);
  // D[row = 4 q + e][column = c]: where the lane's rows go
  uint32_t dst[RT][4];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (MODE == kTall) dst[r][e] = m0 + 16 * r + 4 * q + e;
      else dst[r][e] = my_pairs[min(16 * r + 4 * q + e, rows - 1)];
    }
  w.template owned_block<GC, HALF, false, false>(code, c0 + lr, O, x, xo, nb - 1, nb, lane, smem, smem, lds, ask_scales);
#pragma unroll
  for (int j = 0; j < GC; ++j) {
    const int col = c0 + lr + 16 * j;
    if (col >= O) continue;
    bf16_t* const y = a.m[mat0].y + col;
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (16 * r + 4 * q + e < rows) {
          const float v = w.acc[r][j][e];
          y[(size_t)dst[r][e] * O] = MODE == kGateUp ? swiglu_bf16(v, w.acc[r][CT - 1][e]) : dm_f2bf(v);
        }
  }
}

// One 16 x 16 tile of a riding dense matrix, K a multiple of 2048: sixteen parts of K, the partial tiles added in order, as
// linear.hip's dense_mm_kernel<16, 1> does it (which has a wavefront a part; here it is four) and so with the same bits. As a launch of
// its own that is a chain of 6 us in 16 workgroups (the a / b heads of a gated-delta layer, 51 rows); here it runs beside
// the wide projections' 12288 columns: us, two launches / one, 51 rows 14.6 + 6.3 / 15.3, 600 rows over 4-bit affine weights 62.1 + 6.9 / 64.6.
__device__ __forceinline__ void rider_tile(const Args& a, uint32_t id, uint8_t* smem) {
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, lg = lane >> 4;
  const int rt = (int)(id / (uint32_t)a.d.tiles);
  int t = (int)id - rt * a.d.tiles;
  const int first = (a.d.O[0] + 15) / 16, seg = t >= first;
  t -= seg ? first : 0;
  const bf16_t* w = seg ? a.d.w[1] : a.d.w[0];
  bf16_t* y = seg ? a.d.y[1] : a.d.y[0];
  const int O = seg ? a.d.O[1] : a.d.O[0], col = 16 * t + l16, kw = a.K / 16;
  const bf16_t* xp = a.x + (size_t)min(16 * rt + l16, a.M - 1) * a.K + 8 * lg;
  const bf16_t* wp = w + (size_t)min(col, O - 1) * a.K + 8 * lg;
  f32x4_t acc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < kw; k0 += 128)
#pragma unroll
    for (int h = 0; h < 4; h += 2) {  // (two parts' operands at a time: all four are more registers than the smallest kernel has)
      bf16x8_t xa[2][4], wb[2][4];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int at = (4 * wave + h + i) * kw + k0 + 32 * s;
          xa[i][s] = *reinterpret_cast<const bf16x8_t*>(xp + at);
          wb[i][s] = *reinterpret_cast<const bf16x8_t*>(wp + at);
        }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int s = 0; s < 4; ++s) acc[h + i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[i][s], wb[i][s], acc[h + i], 0, 0, 0);
    }
  f32x4_t* const red = reinterpret_cast<f32x4_t*>(smem) + lane;
#pragma unroll
  for (int i = 0; i < 4; ++i) red[(4 * wave + i) * 64] = acc[i];
  __syncthreads();
  if (wave != 0) return;
  f32x4_t v = red[0];
#pragma unroll
  for (int p = 1; p < 16; ++p) v += red[p * 64];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = 16 * rt + 4 * lg + r;
    if (col < O && row < a.M) y[(size_t)row * O + col] = dm_f2bf(v[r]);
  }
}

// AFF: affine formats, else k-quants; ONE: the kind of every matrix of the launch, or -1. NW wavefronts, K >= 512.
// Plain: grid (column blocks, row tiles); gathered: a workgroup a column block of a tile.
template <bool AFF, int CT, int MODE, int ROWS, int NW, int ONE = -1>
__device__ __forceinline__ void body(const Args& a) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t nmm_smem[];
  int mat0 = 0, cb = blockIdx.x, c0, rows, m0 = 0;
  int64_t row_base = 0;
  const uint32_t* my_pairs = nullptr;
  if constexpr (MODE == kPlain) {
    if ((int)blockIdx.x >= a.blocks) {
      const uint32_t id = (blockIdx.x - (uint32_t)a.blocks) * gridDim.y + blockIdx.y;
      if (id < (uint32_t)a.d.wgs) rider_tile(a, id, nmm_smem);
      return;
    }
#pragma unroll
    for (int i = 1; i < 4; ++i)
      if (i < a.n && (int)blockIdx.x >= a.m[i].cb0) {
        mat0 = i;
        cb = (int)blockIdx.x - a.m[i].cb0;
      }
    m0 = blockIdx.y * ROWS;
    rows = min(ROWS, a.M - m0);
    c0 = cb * (NW / a.ks) * CT * 16;
  } else if constexpr (MODE == kTall) {
    // (a die's workgroups: the row tiles of one column block after the other, so that its L2 fetches the weights once)
    // (the riders first, in whole rounds of dies)
    const uint32_t ahead = ((uint32_t)a.d.wgs + 7u) / 8u * 8u;
    if (blockIdx.x < ahead) {
      if (blockIdx.x < (uint32_t)a.d.wgs) rider_tile(a, blockIdx.x, nmm_smem);
      return;
    }
    const uint32_t id = blockIdx.x - ahead, die = id % 8u, seq = id / 8u, rt = seq % (uint32_t)a.tiles_max;
    cb = (int)(seq / (uint32_t)a.tiles_max * 8u + die);
    if (cb >= a.blocks) return;
#pragma unroll
    for (int i = 1; i < 4; ++i)
      if (i < a.n && cb >= a.m[i].cb0) mat0 = i;
    c0 = (cb - a.m[mat0].cb0) * 128;
    m0 = (int)rt * ROWS;
    rows = min(ROWS, a.M - m0);
  } else {
    // Workgroups go round the eight dies: a tile's column blocks follow each other on one die, whose L2 then fetches
    // the tile's activations once.
    const uint32_t die = blockIdx.x % 8u, seq = blockIdx.x / 8u, tile = seq / (uint32_t)a.blocks * 8u + die;
    c0 = (int)(seq % (uint32_t)a.blocks) * (MODE == kGateUp ? 64 : 128);
    // (all four words in one trip; what lies past the list's end is not used)
    const uint32_t at = min(tile, (uint32_t)a.tiles_max - 1u), n = *a.n_tiles;
    const uint32_t e = __builtin_amdgcn_readfirstlane(a.tile_expert[at]);
    rows = __builtin_amdgcn_readfirstlane((int)a.tile_count[at]);
    my_pairs = a.pair + __builtin_amdgcn_readfirstlane(a.tile_start[at]);
    if (tile >= n) return;
    if ((int)e >= a.E)
      mat0 = 2;
    else
      row_base = (int64_t)e * a.m[0].O;
  }
  const int kind = a.m[mat0].kind;
  auto run = [&](auto kc, auto rc) {
    constexpr int KIND = decltype(kc)::value, RT = decltype(rc)::value;
    if constexpr (MODE == kPlain) tile_body<KIND, RT, CT, ROWS, NW>(a, mat0, c0, rows, m0, nmm_smem);
    else owned_tile<KIND, RT, MODE>(a, mat0, c0, row_base, rows, m0, my_pairs, nmm_smem);
  };
  auto of_kind = [&](auto kc) {
    if (rows <= 16 || ROWS == 16) run(kc, std::integral_constant<int, 1>{});
    else if (rows <= 32 || ROWS == 32) run(kc, std::integral_constant<int, (ROWS >= 32 ? 2 : 1)>{});
    else if (rows <= 48) run(kc, std::integral_constant<int, (ROWS >= 48 ? 3 : 1)>{});
    else run(kc, std::integral_constant<int, (ROWS >= 64 ? 4 : 1)>{});
  };
  if constexpr (ONE >= 0) {
    of_kind(std::integral_constant<int, ONE>{});
  } else if constexpr (AFF) {
    if (kind == kA4) of_kind(std::integral_constant<int, kA4>{});
    else of_kind(std::integral_constant<int, kA8>{});
  } else {
    if (kind == kQ4K) of_kind(std::integral_constant<int, kQ4K>{});
    else of_kind(std::integral_constant<int, kQ6K>{});
  }
}

}  // namespace nmm
