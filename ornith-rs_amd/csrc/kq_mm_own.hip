// The k-quant GEMM of long prompts: Y[M, O] = X[M, K] . W^T, plain or over an expert-sorted pair list, with the
// weights dequantized straight into matrix-core operands by the wavefront that owns their columns.
//
// Replaces, with kq_mm.hip's other forms, kquant::{qmm_t, gather_qmm_t} (/root/reference/src/ops/kquant.rs:783-1027;
// kernels/kquant_mm.h).
//
// A workgroup is four wavefronts, one a SIMD, and a tile of 256 columns by up to 256 rows. A wavefront owns 64 columns over all the rows:
// its weights are dequantized once a tile and never written anywhere, and its 16 x 16 accumulator registers (two column blocks
// by eight row blocks of v_mfma_f32_32x32x16_bf16) are what one wavefront a SIMD leaves room for. The activations, which all
// four wavefronts multiply by, come in slabs of 64 k straight into LDS (global_load_lds, whole 128-byte lines; no registers, no
// writes), three slabs deep, with one barrier a slab that leaves requests in flight. The codes go to LDS the same way, into a
// part that is the wavefront's own: 64 lanes that each read 16 bytes of their own row would look up 64 cache lines a load, whole
// rows of a super-block 8. So do the scales. One super-block is unpacked while the next one's weights travel.
//
// A k step is 16 matrix instructions (at 256 rows), and between them, one piece after each, stands the work for the step
// after: eight fragment reads, the unpacking of two fragments (36 vector instructions of Q4_K, 52 of Q6_K), a slab's
// requests. The order is fixed in the source (sched_barrier after each piece) and every wait for memory is counted by hand. That is
// sound because nothing of it goes to registers: a load to a register in inline assembly is, to the compiler, done there and then, so
// that it may copy or spill what is still to come; and one that it knows of it waits for with everything else in flight.
//
// Shorter prompts (kHalves): tiles of 128 columns by up to 128 rows and two such sets of wavefronts, each over half of K, whose sums meet
// in LDS at the end. With few rows a tile the unpacking is the work, and a wavefront alone on its SIMD issues one instruction every 5
// to 8 clocks (two share 4), so a step of 64 columns costs as much as 8 row blocks' matrix instructions whether there are 2 or 5: half
// the columns a wavefront and twice the wavefronts are 2.2 times as fast a tile (K = 2048, 2 / 4 row blocks 25 / 32 -> 15 / 20 us, K = 4096 42 / 56 -> 23 /
// 30). Four stages of activations with two super-blocks of codes in flight gave nothing, nor did eight wavefronts of 32 columns over
// all of K (K = 4096, 2 row blocks 38).
//
// kThin is one such set, over all of K and two workgroups a compute unit: the sums of the full tile in a fourth of it, for a launch
// that full tiles leave most compute units idle in.
//
// What bounds it: at full size (12288 x 2048, 6621 rows) the matrix cores are busy for 55 % of the launch's clocks. What is left of them are the ways in and
// out of a tile, 3 and 3.5 us of 56 that nothing overlaps, the last of five rounds of tiles (0.88 full), and the step: 0.39 us
// with every compute unit at work where one alone takes 0.29, by the clock, which falls under load; the same loop over weights that are bf16
// already, no vector work at all, is no faster. Below about 160 rows a tile the unpacking (0.14 us a step however few the rows).
//
// Measured on one card, us, launches by themselves, against what this replaces (256 x 128 tiles with weights through LDS): 12288 x 2048 Q4_K at 700 / 1500 /
// 6621 rows 52 / 100 / 342 -> 37 / 74 / 268 (975 -> 1244 TFLOP/s; in a prompt's trace 1135 to 1198), 2048 x 4096 at 6621 132 -> 92, q / k / v (9216 x 2048 Q6_K) at
// 700 / 6621 44 / 292 -> 37 / 229; the experts of 6621 tokens, 256 of them, against tiles of 192 and 64 rows with activations through registers: gate or up 151 -> 107
// with 207 rows each, 148 -> 120 with a spread as a router's, down (K = 512) 272 -> 186 and 256 -> 219. In a trace of that prompt: gate or up 131, down 227, router +
// shared gate + up 46. With kHalves, against the few-row kernels and kFour: 12288 x 2048
// Q4_K at 129 / 200 rows 25 / 25 -> 18 / 20, 2048 x 4096 Q4_K at 600 / 1200 / 2000 30 / 44 / 46 -> 25 / 29 / 39, Q6_K 36 / 53 / 55 -> 28 / 33 / 42.
#include <type_traits>

#include "kq_mm_own.h"

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

template <int N>
using IC = std::integral_constant<int, N>;
template <class F, int... I>
__device__ __forceinline__ void each_of(F f, std::integer_sequence<int, I...>) {
  (f(IC<I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void each(F f) {
  each_of(f, std::make_integer_sequence<int, N>{});
}

// ---- requests, all of them to LDS: waited for by count (the compiler does not connect them with the reads of what they bring)
template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// BYTES (2, 4 or 16) a lane from a base the wavefront shares and the lane's offset to LDS, the lanes' pieces side by side at `lds` (two bytes
// in places of four)
template <int BYTES>
__device__ __forceinline__ void dma(const uint8_t* base, uint32_t off, uint32_t lds) {
  typedef const __attribute__((address_space(1))) void glb_t;
  typedef __attribute__((address_space(3))) void lds_t;
  static_assert(BYTES == 2 || BYTES == 4 || BYTES == 16, "");
  if constexpr (BYTES == 16) __builtin_amdgcn_global_load_lds((glb_t*)(uint64_t)(base + off), (lds_t*)(uint64_t)lds, 16, 0, 0);
  else if constexpr (BYTES == 4) __builtin_amdgcn_global_load_lds((glb_t*)(uint64_t)(base + off), (lds_t*)(uint64_t)lds, 4, 0, 0);
  else __builtin_amdgcn_global_load_lds((glb_t*)(uint64_t)(base + off), (lds_t*)(uint64_t)lds, 2, 0, 0);
}
__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return (uint32_t)(uint64_t)(const __attribute__((address_space(3))) void*)p;
}
__device__ __forceinline__ const uint8_t* uniform(const uint8_t* p) {
  const uint64_t v = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return dm_global_ptr<const uint8_t>(((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ void barrier_only() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// ---- the weights of 32 rows (a wavefront's column block) and one super-block ---------------------
// The codes go to LDS as whole rows of the super-block (kInstr requests of 64 16-byte pieces), piece `at(row, p)` of a row at a
// place that keeps the rows of a fragment on different banks; a lane then takes the pieces of its row that are its own.
template <int KIND>
struct Fmt;
template <>
struct Fmt<ORNITH_Q4K> {
  static constexpr int kQ = 128, kS = 12, kD = 4, kInstr = 4, kHalf = 2;
  static __device__ __forceinline__ void source(int n, int& row, int& p) {  // what lies at 16-byte place n
    row = n >> 3;
    p = (n & 7) ^ ((row >> 1) & 7);
  }
  static __device__ __forceinline__ int at(int row, int p) { return 16 * (8 * row + (p ^ ((row >> 1) & 7))); }
  // piece I of half HF that lane half h takes: bytes 16 h .. of 64-group 2 HF + I
  static __device__ __forceinline__ int piece(int hf, int i, int h) { return 2 * (2 * hf + i) + h; }
};
template <>
struct Fmt<ORNITH_Q6K> {
  static constexpr int kQ = 192, kS = 16, kD = 2, kInstr = 6, kHalf = 3;
  static __device__ __forceinline__ void source(int n, int& row, int& p) {
    row = n / 12;
    p = n - 12 * row - ((row >> 2) & 3);
    p += p < 0 ? 12 : 0;
  }
  static __device__ __forceinline__ int at(int row, int p) {
    int j = p + ((row >> 2) & 3);
    j -= j >= 12 ? 12 : 0;
    return 16 * (12 * row + j);
  }
  // low rows a and b (I = 0, 1) and high bits (2) of half HF
  static __device__ __forceinline__ int piece(int hf, int i, int h) { return i < 2 ? 4 * hf + 2 * i + h : 8 + 2 * hf + h; }
};
// The scales of a super-block, four words a column: of Q4_K its 12 bytes of scales and, fourth, d and dmin; of Q6_K its 16 bytes of
// scales, and d in a request by itself. A request brings them of 16 columns, a word a lane.
template <int KIND, int TN>
struct Sc {
  typedef Fmt<KIND> F;
  static constexpr int kReq = 2 * TN + (KIND == ORNITH_Q6K);
  u32x4_t sc;
  uint32_t d;  // Q6_K
  // of column l32 of block j
  __device__ __forceinline__ void read(const uint8_t* lds, int j, int l32) {
    sc = *reinterpret_cast<const u32x4_t*>(lds + 16 * (32 * j + l32));
    if constexpr (KIND == ORNITH_Q6K) d = *reinterpret_cast<const uint16_t*>(lds + 512 * TN + 4 * (32 * j + l32));
  }
  __device__ __forceinline__ uint32_t dm() const {
    if constexpr (KIND == ORNITH_Q4K) return sc[3];
    else return d;
  }
};

// the upper half of a's lanes trades places with the lower half of b's (swap16: a's odd rows of sixteen with b's even ones)
__device__ __forceinline__ u32x2_t swap32(uint32_t a, uint32_t b) {
  const auto v = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  return u32x2_t{v[0], v[1]};
}
__device__ __forceinline__ u32x2_t swap16(uint32_t a, uint32_t b) {
  const auto v = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  return u32x2_t{v[0], v[1]};
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

// w >> N (N < 0: w << -N), another instruction in every step TAG: merged into one, shifted words would be kept from step to step
template <int N, int TAG>
__device__ __forceinline__ uint32_t shifted(uint32_t w) {
  uint32_t r;
  if constexpr (N >= 0)
    asm("v_lshrrev_b32 %0, %1, %2 ; %3" : "=v"(r) : "n"(N), "v"(w), "n"(TAG));
  else
    asm("v_lshlrev_b32 %0, %1, %2 ; %3" : "=v"(r) : "n"(-N), "v"(w), "n"(TAG));
  return r;
}

// The operand of k step T (0 .. 15 of the super-block), made in seven pieces so that they can stand between matrix instructions.
template <int KIND>
struct Deq {
  typedef Fmt<KIND> F;
  u32x4_t q[2 * F::kHalf];  // the lane's codes, by half
  float dl, dh, nm;         // d * 2^24, d * 2^20, -dmin
  uint32_t sc4, m4;         // the half's four scales and minima
  float s, o;
  uint32_t e0, o0, e1, o1;
  float x0, x1;
  u32x4_t f;
  template <int T, int P, class Z>
  __device__ __forceinline__ void piece(const Z& z, int h) {
    constexpr int HF = T >> 3, QD = (T >> 1) & 3, NIB = KIND == ORNITH_Q4K ? QD & 1 : QD >> 1;
    if constexpr (P == 0) {
      if constexpr (KIND == ORNITH_Q4K) {
        if constexpr (T == 0) {
          const float d = dm_h2f((f16_t)(z.dm() & 0xffffu));
          dl = d * 16777216.f;
          dh = d * 1048576.f;
          nm = -dm_h2f((f16_t)(z.dm() >> 16));
          sc4 = z.sc[0] & 0x3f3f3f3fu;
          m4 = z.sc[1] & 0x3f3f3f3fu;
        }
        if constexpr (T == 8) {
          sc4 = (z.sc[2] & 0x0f0f0f0fu) | ((z.sc[0] & 0xc0c0c0c0u) >> 2);
          m4 = ((z.sc[2] >> 4) & 0x0f0f0f0fu) | ((z.sc[1] & 0xc0c0c0c0u) >> 2);
        }
        if constexpr (T % 2 == 0) {
          s = (NIB ? dh : dl) * dm_ubyte<QD>(sc4);
          o = nm * dm_ubyte<QD>(m4);
        }
      } else {
        if constexpr (T == 0) dl = dm_h2f((f16_t)z.dm());
        if constexpr (T % 2 == 0) {  // scale 8 HF + 2 QD + h of the sixteen
          const float v = dl * (float)(int)(int8_t)(((z.sc[T >> 2] >> (8 * h)) >> (16 * (QD & 1))) & 0xffu);
          s = v * (NIB ? 1048576.f : 16777216.f);
          o = -32.f * v;
        }
      }
    } else if constexpr (P == 1 || P == 2) {
      constexpr int I = P - 1, W = 2 * (T & 1) + I;
      constexpr uint32_t M = NIB ? 0x00f000f0u : 0x000f000fu;
      uint32_t e, od;
      if constexpr (KIND == ORNITH_Q4K) {
        const uint32_t w = q[T >> 2][W];
        e = w & M;
        od = shifted<8, T>(w) & M;
      } else {
        constexpr int SH = 4 - 2 * (QD & 1);
        constexpr uint32_t MH = NIB ? 0x03000300u : 0x00300030u;
        const uint32_t w = q[3 * HF + (QD & 1)][W], hb = q[3 * HF + 2][W];
        e = (w & M) | (shifted<-SH, T>(hb) & MH);
        od = (shifted<8, T>(w) & M) | (shifted<8 - SH, T>(hb) & MH);
      }
      if constexpr (I == 0) e0 = e, o0 = od;
      else e1 = e, o1 = od;
    } else if constexpr (P == 3) {
      x0 = fma_half<0>(s, e0, o), x1 = fma_half<0>(s, o0, o);
    } else if constexpr (P == 4) {
      const float y0 = fma_half<1>(s, e0, o), y1 = fma_half<1>(s, o0, o);
      f[0] = dm_f2bf2(x0, x1);
      x0 = y0, x1 = y1;
    } else if constexpr (P == 5) {
      const float y0 = fma_half<0>(s, e1, o), y1 = fma_half<0>(s, o1, o);
      f[1] = dm_f2bf2(x0, x1);
      x0 = y0, x1 = y1;
    } else {
      const float y0 = fma_half<1>(s, e1, o), y1 = fma_half<1>(s, o1, o);
      f[2] = dm_f2bf2(x0, x1);
      f[3] = dm_f2bf2(y0, y1);
    }
  }
};

// How a workgroup's wavefronts divide its tile: four of 64 columns, four of 32, or two sets of four of 32 columns that have half of K each
enum { kFour, kThin, kHalves };
constexpr int tn_of(int form) { return form == kFour ? 2 : 1; }
constexpr int sets_of(int form) { return form == kHalves ? 2 : 1; }
constexpr int threads_of(int form) { return 256 * sets_of(form); }
constexpr int cols_of(int form) { return form == kFour ? kOwnCols : 128; }
constexpr int rows_of(int form) { return form == kFour ? kOwnRows : 128; }

constexpr int kStages = 3;  // of 64 k: 128 bytes of a row
// LDS: a set's activations, then a part for each wavefront's codes and one for its scales (Q6_K's d in a request of 64 words, half of them unused with
// 32 columns). kThin has 77 KB, so that a compute unit holds two workgroups.
constexpr int acts_of(int form) { return kStages * rows_of(form) * 128; }
constexpr int codes_of(int form) { return 32 * tn_of(form) * 192; }
constexpr int scales_of(int form) { return 512 * tn_of(form) + 256; }
constexpr int lds_of(int form) { return sets_of(form) * (acts_of(form) + 4 * (codes_of(form) + scales_of(form))); }

template <int KIND, int TM, int FORM, bool GATHER>
__device__ __forceinline__ void own_tile(const OwnArgs& a, const OwnMat& mt, uint8_t* smem, int n0, int rows, int m0,
                                         int64_t wrow0, const uint32_t* pairs) {
  typedef Fmt<KIND> F;
  constexpr int TN = tn_of(FORM), STAGE = TM * 4096, SL = TN * TM;
  constexpr int CODES = sets_of(FORM) * acts_of(FORM), SCALES = CODES + 4 * sets_of(FORM) * codes_of(FORM);  // where in LDS
  typedef Sc<KIND, TN> Z;
  constexpr int NC = TN * F::kInstr + Z::kReq;  // requests of a super-block's weights
  const int tid = threadIdx.x, lane = tid & 63, wave_of = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, h = lane >> 5;
  const int wave = wave_of & 3, set = wave_of >> 2, row_blocks = a.K >> 8, nb = FORM == kHalves ? row_blocks / 2 : row_blocks, b0 = set * nb;
  uint32_t qo[TN][F::kInstr];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int r0 = n0 + 32 * TN * wave + 32 * j;
#pragma unroll
    for (int i = 0; i < F::kInstr; ++i) {
      int row, p;
      F::source(64 * i + lane, row, p);
      qo[j][i] = (uint32_t)min(r0 + row, mt.O - 1) * (uint32_t)(row_blocks * F::kQ) + 16 * p;
    }
  }
  const uint8_t *qb = uniform(mt.qs + (wrow0 * row_blocks + b0) * F::kQ), *sb = uniform(mt.scales + (wrow0 * row_blocks + b0) * F::kS),
                *db = uniform(mt.dm + (wrow0 * row_blocks + b0) * F::kD);
  const int word = lane & 3;
  const bool of_d = KIND == ORNITH_Q4K && word == 3;
  const uint8_t* sp[2 * TN];  // what the lane takes of 16 columns' scales
#pragma unroll
  for (int i = 0; i < 2 * TN; ++i) {
    const uint32_t row = (uint32_t)min(n0 + 32 * TN * wave + 16 * i + (lane >> 2), mt.O - 1) * (uint32_t)row_blocks;
    sp[i] = of_d ? db + row * F::kD : sb + (row * F::kS + 4 * word);
  }
  const uint32_t sp_step = of_d ? F::kD : F::kS;
  const uint32_t dof = (uint32_t)min(n0 + 32 * TN * wave + (TN == 2 ? lane : l32), mt.O - 1) * (uint32_t)row_blocks * F::kD;  // Q6_K
  __builtin_amdgcn_sched_barrier(0);
  // request i of a slab's activations: eight rows of row block i, 128 bytes each
  uint32_t* const s_dst = reinterpret_cast<uint32_t*>(smem + lds_of(FORM));  // (gathered form)
  uint32_t* const s_src = s_dst + kOwnRows;
  uint32_t pr[TM];
  if constexpr (GATHER) {  // (the rows a wavefront asks for, eight of each block, go to a part of its own)
    const uint8_t* pb = uniform((const uint8_t*)pairs);
    dma<4>(pb, 4 * min(tid, rows - 1), lds_address(s_dst) + 256 * wave);
    dma<4>(pb, 4 * min(32 * (lane >> 3) + 8 * wave + (lane & 7), rows - 1), lds_address(s_src) + 256 * wave);
  } else {
#pragma unroll
    for (int i = 0; i < TM; ++i) pr[i] = m0 + min(32 * i + 8 * wave + (lane >> 3), rows - 1);
  }
  uint8_t* const mine = smem + CODES + wave_of * (32 * TN * F::kQ);
  const uint8_t* const my_scales = smem + SCALES + wave_of * scales_of(FORM);
  const uint32_t mine_at = lds_address(mine), scales_at = lds_address(my_scales);
  Z z[TN];
  // request I of a super-block's weights: the first (NEXT = 0), or the one after what was asked for before
  auto weights = [&](auto next, auto ic) {
    constexpr int NEXT = decltype(next)::value, I = decltype(ic)::value, J = I - TN * F::kInstr;
    if constexpr (I < TN * F::kInstr) dma<16>(qb + NEXT * F::kQ, qo[I / F::kInstr][I % F::kInstr], mine_at + 1024 * I);
    else if constexpr (J < 2 * TN) {
      sp[J] += NEXT * sp_step;
      dma<4>(sp[J], 0, scales_at + 256 * J);
    } else dma<2>(db + NEXT * F::kD, dof, scales_at + 512 * TN);
  };
  each<NC>([&](auto ic) { weights(IC<0>{}, ic); });
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (GATHER) {
    wait_loads<NC>();
#pragma unroll
    for (int i = 0; i < TM; ++i) pr[i] = s_src[64 * wave + 8 * i + (lane >> 3)];
  }
  uint32_t xo[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const uint32_t src = GATHER && a.up_div > 1 ? dm_div(pr[i], (uint32_t)a.up_div, a.up_magic) : pr[i];
    xo[i] = src * (2u * (uint32_t)a.K) + 16 * ((lane & 7) ^ ((4 * wave + (lane >> 4)) & 7));
  }
  const uint8_t* xg = reinterpret_cast<const uint8_t*>(a.x) + 512 * b0;
  const uint32_t mem = set * acts_of(FORM), at = lds_address(smem) + mem + wave * 1024;
#pragma unroll
  for (int s = 0; s < kStages; ++s)
#pragma unroll
    for (int i = 0; i < TM; ++i) dma<16>(xg + 128 * s, xo[i], at + s * STAGE + i * 4096);
  __builtin_amdgcn_sched_barrier(0);
  f32x16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  // step T's fragment of row block i: piece 4 ((T >> 1) & 1) + 2 h + (T & 1) of the slab's 128 bytes, which lie turned by the row
  uint32_t rd[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) rd[t] = mem + l32 * 128 + 16 * ((4 * (t >> 1) + 2 * h + (t & 1)) ^ ((l32 >> 1) & 7));
  uint32_t st = 0;  // stage of the slab
  auto after = [](uint32_t s) { return s == 2 * STAGE ? 0u : s + STAGE; };
  bf16x8_t af[TM], bf[2][TN];
  auto read = [&](auto tc, uint32_t from, int i) {
    af[i] = *reinterpret_cast<const bf16x8_t*>(smem + (rd[decltype(tc)::value & 3] + from) + i * 4096);
  };
  Deq<KIND> dq[TN];
  auto codes = [&](auto hc, int j) {
    constexpr int HF = decltype(hc)::value;
#pragma unroll
    for (int i = 0; i < F::kHalf; ++i)
      dq[j].q[F::kHalf * HF + i] = *reinterpret_cast<const u32x4_t*>(mine + j * (32 * F::kQ) + F::at(l32, F::piece(HF, i, h)));
  };
  wait_loads<2 * TM>();  // the weights and stage 0
  barrier_only();
#pragma unroll
  for (int j = 0; j < TN; ++j) z[j].read(my_scales, j, l32), codes(IC<0>{}, j), codes(IC<1>{}, j);
#pragma unroll
  for (int i = 0; i < TM; ++i) read(IC<0>{}, st, i);
  each<TN * 7>([&](auto pc) {
    constexpr int J = decltype(pc)::value / 7, P = decltype(pc)::value % 7;
    dq[J].template piece<0, P>(z[J], h);
  });
#pragma unroll
  for (int j = 0; j < TN; ++j) bf[0][j] = __builtin_bit_cast(bf16x8_t, dq[j].f);
  __builtin_amdgcn_sched_barrier(0);

  for (int ib = 0; ib < nb; ++ib) {
    // A slab's activations are asked for three slabs ahead (into the stage it leaves), the next block's weights in slab 0
    // (the wavefront's own part of LDS has been read by then).
    const bool last = ib + 1 == nb;
    each<16>([&](auto tc) {
      constexpr int T = decltype(tc)::value, S = T >> 2, U = T + 1;  // U: the step being made ready
      const uint32_t st1 = after(st);
      if constexpr ((T & 3) == 3) {
        // Slab S + 1 has arrived (asked for two slabs ago: a slab's requests, in slab 1 the weights' too, may be out behind it),
        // in slab 2 the weights; everyone has read what slab S holds
        if constexpr (S == 0 || S == 3) wait_loads<TM>();
        if constexpr (S == 1) {
          if (last) wait_loads<TM>();
          else wait_loads<TM + NC>();
        }
        if constexpr (S == 2) {
          if (last) wait_loads<0>();
          else wait_loads<TM>();
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        barrier_only();
      }
      each<SL>([&](auto ic) {
        constexpr int I = decltype(ic)::value, M = I / TN, N = I % TN;
        acc[M][N] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bf[T & 1][N], af[M], acc[M][N], 0, 0, 0);
        if constexpr (N == TN - 1) read(IC<U>{}, (T & 3) == 3 ? st1 : st, M);
        if constexpr ((T == 12 || T == 15) && I < TN) codes(IC<(T == 12 ? 0 : 1)>{}, I);
        if constexpr (T == 14 && I < TN) z[I].read(my_scales, I, l32);  // (the last that step 13 needed)
        constexpr int P0 = I * (TN * 7) / SL, P1 = (I + 1) * (TN * 7) / SL;
        each<P1 - P0>([&](auto pc) {
          constexpr int Q = P0 + decltype(pc)::value, J = Q % TN, P = Q / TN;
          dq[J].template piece<(U & 15), P>(z[J], h);
          if constexpr (P == 6) bf[U & 1][J] = __builtin_bit_cast(bf16x8_t, dq[J].f);
        });
        if constexpr ((T & 3) == 3) {
          constexpr int NR = TM + (S == 0 ? NC : 0);
          if constexpr ((I * NR + SL - 1) / SL < ((I + 1) * NR + SL - 1) / SL)
            each<NR>([&](auto nc) {
              constexpr int Q = decltype(nc)::value;
              if constexpr (Q * SL / NR == I) {
                if constexpr (Q < TM) {
                  if (S == 0 || !last) dma<16>(xg + 128 * (S + 3), xo[Q], at + st + Q * 4096);
                } else {
                  if (!last) weights(IC<1>{}, IC<Q - TM>{});
                }
              }
            });
        }
        __builtin_amdgcn_sched_barrier(0);
      });
      if constexpr ((T & 3) == 3) st = st1;
    });
    xg += 512;
    qb += F::kQ;
    db += F::kD;
  }
  if constexpr (FORM == kHalves) {
    // each set finishes every other row block, and hands the other its part of the rest
    barrier_only();
    f32x4_t* const part = reinterpret_cast<f32x4_t*>(smem) + (size_t)wave * TM * 256 + lane;
#pragma unroll
    for (int i = 0; i < TM; ++i)
      if ((i & 1) != set)
#pragma unroll
        for (int e = 0; e < 4; ++e) part[i * 256 + e * 64] = f32x4_t{acc[i][0][4 * e], acc[i][0][4 * e + 1], acc[i][0][4 * e + 2], acc[i][0][4 * e + 3]};
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    barrier_only();
#pragma unroll
    for (int i = 0; i < TM; ++i)
      if ((i & 1) == set)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const f32x4_t v = part[i * 256 + e * 64];
#pragma unroll
          for (int f = 0; f < 4; ++f) acc[i][0][4 * e + f] += v[f];
        }
  }
  // D[n = 8 b + 4 h + r][m = l32]: two swaps of lanes bring 32 columns of a row into four lanes, 16 bytes each
  const int half = 16 * ((lane >> 4) & 1) + 8 * h;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    if (FORM == kHalves && (i & 1) != set) continue;
    bf16_t* y[2];
    bool live[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int r = 32 * i + 16 * b + (lane & 15);
      live[b] = r < rows;
      y[b] = mt.y + (size_t)(GATHER ? s_dst[r] : (uint32_t)(m0 + r)) * mt.O + n0 + 32 * TN * wave + half;
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const f32x16_t& c = acc[i][j];
      u32x4_t v[2];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const u32x2_t p = swap32(dm_f2bf2(c[8 * b], c[8 * b + 1]), dm_f2bf2(c[8 * b + 4], c[8 * b + 5]));
        const u32x2_t q = swap32(dm_f2bf2(c[8 * b + 2], c[8 * b + 3]), dm_f2bf2(c[8 * b + 6], c[8 * b + 7]));
        v[b] = u32x4_t{p[0], q[0], p[1], q[1]};  // columns 16 b + 8 h ..
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const u32x2_t p = swap16(v[0][e], v[1][e]);
        v[0][e] = p[0];
        v[1][e] = p[1];
      }
      const int left = mt.O - (n0 + 32 * TN * wave + 32 * j + half);
#pragma unroll
      for (int b = 0; b < 2; ++b)
        if (live[b] && left > 0) {
          // (16 bytes a lane whatever the alignment of y's rows: eight pieces of 2 bytes, which lie apart in memory from lane to lane, made 131 x 512, 16
          // experts of 207 rows, 12.3 us, this way 9.5, and 12291 x 512 at 2049 rows 83, this way 48)
          if (left >= 8) __builtin_memcpy(y[b] + 32 * j, &v[b], 16);
          else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
              if (e < left) y[b][32 * j + e] = (bf16_t)(v[b][e >> 1] >> (16 * (e & 1)));
          }
        }
    }
  }
}

constexpr int kMixed = 2;  // the matrices of the launch differ in kind
template <int KIND, int FORM, bool GATHER>
__global__ __launch_bounds__(threads_of(FORM)) __attribute__((amdgpu_waves_per_eu(FORM == kFour ? 1 : 2, FORM == kFour ? 1 : 2))) void kq_mm_own_kernel(OwnArgs a) {
  // (one array: with more than one, the compiler does connect some reads with requests, and waits for everything in flight ahead of them)
  __shared__ __attribute__((aligned(1024))) uint8_t smem[lds_of(FORM) + (GATHER ? 4 * (kOwnRows + 256) : 0)];
  int rows, m0 = 0, tc, mat = 0;
  int64_t wrow0 = 0;
  const uint32_t* pairs = nullptr;
  const uint32_t die = blockIdx.x & 7, seq = blockIdx.x >> 3;
  if constexpr (GATHER) {
    // The columns over a plan's tile stay on one die, whose cache its rows then stay in. kThin: first all tiles' upper 128 rows, then the lower ones, which
    // not every tile has, four dies on (taken in turn they fall on every other die, and half the dies idle: 512 x 4352, 64 experts of 207 rows, round
    // the dies column by column 145 us, in turn 96)
    const uint32_t eights = ((uint32_t)a.tiles_max + 7u) / 8u, at8 = seq / (uint32_t)a.col_tiles;
    const uint32_t sub = FORM == kThin && at8 >= eights ? 1u : 0u, tile = (at8 - sub * eights) * 8u + ((die + 4u * sub) & 7u);
    const uint32_t at = min(tile, (uint32_t)a.tiles_max - 1u), n = *a.n_tiles;
    tc = (int)(seq % (uint32_t)a.col_tiles);
    const uint32_t e = __builtin_amdgcn_readfirstlane(a.tile_expert[at]);
    rows = __builtin_amdgcn_readfirstlane((int)a.tile_count[at]);
    pairs = a.pair + __builtin_amdgcn_readfirstlane(a.tile_start[at]);
    if (tile >= n) return;
    if (a.expert_at) {
      // a plan of lower tiles (16, 32 or 64 rows): the first of as many as a tile here holds works on the pairs of them all
      const int first = (int)__builtin_amdgcn_readfirstlane(a.expert_at[e]), st = (int)(pairs - a.pair);
      const int end = (int)e + 1 < a.E ? (int)__builtin_amdgcn_readfirstlane(a.expert_at[e + 1]) : a.M;
      if ((st - first) % kOwnRows != 0) return;
      rows = min(end - st, kOwnRows);
    }
    if constexpr (FORM == kThin) {
      rows = min(rows - (int)(sub * 128), 128);
      if (rows <= 0) return;
      pairs += sub * 128;
    }
    wrow0 = (int64_t)e * a.m[0].O;
  } else {
    const int total = a.row_tiles * a.col_tiles, per = (total + 7) / 8, id = (int)die * per + (int)seq;
    if ((int)seq >= per || id >= total) return;
    constexpr int GM = 8;
    const int grp = id / (GM * a.col_tiles), in = id - grp * GM * a.col_tiles, gm = min(GM, a.row_tiles - grp * GM);
    m0 = (grp * GM + in % gm) * a.tile_rows;
    tc = in / gm;
    rows = min(a.tile_rows, a.M - m0);
#pragma unroll
    for (int i = 1; i < 4; ++i)
      if (i < a.n && tc >= a.m[i].t0) mat = i;
  }
  const OwnMat mt = a.m[mat];
  const int n0 = (tc - mt.t0) * cols_of(FORM);
  const int groups = (rows + 31) >> 5;
  auto of_kind = [&](auto kc) {
    constexpr int KD = decltype(kc)::value;
#define OWN(N) own_tile<KD, N, FORM, GATHER>(a, mt, smem, n0, rows, m0, wrow0, pairs)
    if constexpr (FORM == kFour) {
      if (groups >= 8) return OWN(8);
      if (groups == 7) return OWN(7);
      if (groups == 6) return OWN(6);
      if (groups == 5) return OWN(5);
    }
    if (groups >= 4) OWN(4);
    else if (groups == 3) OWN(3);
    else OWN(2);
#undef OWN
  };
  if constexpr (KIND != kMixed) of_kind(IC<KIND>{});
  else if (mt.kind == ORNITH_Q4K) of_kind(IC<ORNITH_Q4K>{});
  else of_kind(IC<ORNITH_Q6K>{});
}

}  // namespace

bool kq_mm_own_ok(const ornith_kmatrix& w, const void* x, size_t rows) {
  return w.K >= 256 && w.K % 256 == 0 && rows * w.K * 2 < (size_t(1) << 32) && (size_t)w.O * (w.K / 256) * 192 < (size_t(1) << 32) &&
         (((uintptr_t)x | (uintptr_t)w.d_qs) & 15) == 0 && (((uintptr_t)w.d_scales | (uintptr_t)w.d_dm) & 3) == 0;
}

// What the few-row kernels don't take (up to the lines of mm_narrow_host.h, where their splits suit better) runs here from 129 rows on. us, kq_mm.hip's
// 128-row tiles / here, Q4_K at 129 rows: 264 x 512 9.2 / 6.2, 264 x 2048 28 / 15, 2560 x 2048 28 / 13, 8192 x 4096 53 / 24.
bool kq_mm_own_suits(const ornith_kmatrix& w, const void* x, int M) { return ornith_option_gemm_duo() && M > 128 && kq_mm_own_ok(w, x, M); }

// ... and those that do it in kHalves, one matrix at a time whatever shares the launch, for the sums' order: up to the rows at which the widest launches that
// bring it (12288 columns, 2048 with a few more) are one round of its tiles, so that none of them is split in two. us, kFour / kHalves: 8192 + 4096 columns of K = 2048, Q4_K,
// 200 / 256 / 300 rows 25 / 20, 27 / 21, 27 / 32; 2048 x 4096 Q4_K at 1500 / 2000 / 2400 rows 43 / 32, 46 / 39, 47 / 53. A matrix in between, whose own tiles would be one round for
// longer, has kThin past that (4096 x 2048 at 300 rows 14 here, 16 there). Up to 512 columns are left to the launch of the wide matrices beside them;
// up to 2048 of K < 2048 are as fast in kThin and faster together in kFour (four of 2048 x 512 at 1025 / 2000 rows 20 / 30 here, 15 / 22 there).
bool kq_mm_own_halves(const ornith_kmatrix& w, int M) {
  return w.K % 512 == 0 && (w.O > 2048 ? M <= 256 : w.O > 512 && w.K >= 2048 && M <= 2048);
}

OwnMat kq_mm_own_mat(const ornith_kmatrix& w, void* y) {
  return {(const uint8_t*)w.d_qs, (const uint8_t*)w.d_scales, (const uint8_t*)w.d_dm, (bf16_t*)y, w.O, w.kind, 0};
}

// A plain launch's form. kFour and kThin give the same sums, so what shares a launch may decide between them: kThin while its tiles are
// one a compute unit, as kFour leaves three of four idle then and its tile takes half as long again. us, kFour / kThin, Q4_K: 2560 x 2048 at 300 / 600 / 1200
// rows 23 / 16, 23 / 16, 24 / 21, 3072 x 4096 at 600 43 / 28; past that (320 tiles) level: 2048 x 2600 x 2048 28 / 28, 8192 x 600 x 4096 52 / 56. Of few slabs
// the ways in and out weigh most, and two workgroups a compute unit hide one another's: K = 512, 320 / 512 tiles, Q4_K 12 / 11, 14 / 13, Q6_K 13 / 12, 15 / 14.
bool kq_mm_own_thin(const OwnArgs& a, int units) {
  long tiles = 0;
  for (int i = 0; i < a.n; ++i) tiles += (long)((a.m[i].O + 127) / 128) * ((a.M + 127) / 128);
  return tiles <= (a.K <= 512 ? 2L : 1L) * units;
}

// ... and a gathered one's (the tiles are in the device's hands: what the host knows of them is the experts' mean), while kFour would leave half the compute units
// idle and more. us, Q4_K, kFour / kThin, rows an expert: 2048 x 512, 8 experts of 128 / 300 13 / 9.1, 19 / 11, 16 of 207 19 / 19, 32 of 128 19 / 22;
// 512 x 2048, 16 experts of 128 45 / 21, 64 of 80 / 207 34 / 28, 49 / 51, 128 of 80 42 / 49; 512 x 4352, 16 of 207 87 / 42, 64 of 128 91 / 76.
bool kq_mm_own_thin_experts(int O, int E, int pairs, int units) {
  return 2L * E * ((pairs / E + kOwnRows - 1) / kOwnRows) * ((O + kOwnCols - 1) / kOwnCols) <= units;
}

int kq_mm_own(ornith_ctx* ctx, OwnArgs& a, bool gather) {
  int kind = a.m[0].kind, grid, threads = 256;
  typedef void (*Kernel)(OwnArgs);
  Kernel k;
  if (gather) {
    a.up_magic = dm_div_magic(a.up_div);
    const bool thin = kq_mm_own_thin_experts(a.m[0].O, a.E, a.M, ctx->compute_units);
    const int cols = cols_of(thin ? kThin : kFour);
    a.col_tiles = (a.m[0].O + cols - 1) / cols;
    grid = a.col_tiles * ((a.tiles_max + 7) / 8 * 8) * (thin ? 2 : 1);
    k = kind == ORNITH_Q4K ? (thin ? kq_mm_own_kernel<ORNITH_Q4K, kThin, true> : kq_mm_own_kernel<ORNITH_Q4K, kFour, true>)
                           : (thin ? kq_mm_own_kernel<ORNITH_Q6K, kThin, true> : kq_mm_own_kernel<ORNITH_Q6K, kFour, true>);
  } else {
    // Tile height: a tile takes about as long as 6 + its row blocks (kFour; K = 2048, one tile a compute unit, us: 8 blocks 53, 7 49, 6 44,
    // 5 42; K = 4096 8 82, 5 61, 2 42), in the same measure 2.7 + 0.675 of them (kHalves; K = 2048 2 blocks 15, 3 18, 4 20; K = 4096 23, 27, 30; kThin 15, 19, 22;
    // 27, 33, 37), and the rounds of tiles count.
    const int form = a.halves ? kHalves : kq_mm_own_thin(a, ctx->compute_units) ? kThin : kFour;
    threads = threads_of(form);
    a.col_tiles = 0;
    for (int i = 0; i < a.n; ++i) {
      a.m[i].t0 = a.col_tiles;
      a.col_tiles += (a.m[i].O + cols_of(form) - 1) / cols_of(form);
      if (a.m[i].kind != kind) kind = kMixed;
    }
    long best = 0;
    for (int tm = rows_of(form) / 32; tm >= 2; --tm) {
      const long tiles = (long)((a.M + 32 * tm - 1) / (32 * tm)) * a.col_tiles, rounds = (tiles + ctx->compute_units - 1) / ctx->compute_units;
      const long cost = rounds * (form == kFour ? 6 + tm : 4 + tm);
      if (best == 0 || cost < best) best = cost, a.tile_rows = 32 * tm;
    }
    a.row_tiles = (a.M + a.tile_rows - 1) / a.tile_rows;
    grid = (a.row_tiles * a.col_tiles + 7) / 8 * 8;
#define OWN(F) (kind == kMixed ? kq_mm_own_kernel<kMixed, F, false> : kind == ORNITH_Q4K ? kq_mm_own_kernel<ORNITH_Q4K, F, false> : kq_mm_own_kernel<ORNITH_Q6K, F, false>)
    k = form == kFour ? OWN(kFour) : form == kThin ? OWN(kThin) : OWN(kHalves);
#undef OWN
  }
  hipLaunchKernelGGL(k, dim3(grid), dim3(threads), 0, ctx->stream, a);
  ORN_LAUNCH_CHECK("kq_mm_own_kernel");
  return ORNITH_OK;
}
