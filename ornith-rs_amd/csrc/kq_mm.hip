// Q4_K / Q6_K tiled GEMM on the matrix cores, for prefill widths.
//
// Replaces kquant::{qmm_t, gather_qmm_t, matmul, gather_matmul}
// (/root/reference/src/ops/kquant.rs:783-1027; kernels/kquant_mm.h): Y[M,O] = X[M,K] . W^T
// with the weight tile dequantized to bf16 on the way into LDS and fp32 accumulation, and
// the expert-gathered form where each tile's rows belong to one routed expert.
//
// This is the one GEMM-shaped piece of the path (81 % of a prefill chunk in the
// reference, /root/reference/src/bin/arithmetic.rs:4-7), so it runs on MFMA
// (v_mfma_f32_32x32x16_bf16), the weights read as k-quant codes (the 144 / 210 bytes per 256
// weights that HBM holds) and dequantized with the arithmetic of kquant::dequantize
// (d*sc*q - dmin*m, resp. d*sc*q), rounded to bf16. Here are the dispatch, the expert-sorted pair list and the
// form for any shape and alignment, and for what the options take off the others: a workgroup tile of BM x 128 outputs over K slabs of 128; activations go
// global -> LDS as they are, weights are dequantized on the way into LDS; LDS rows padded by
// 8 elements so the 16-byte fragment reads of 32 consecutive rows spread over the banks;
// four wavefronts: 2 x 2 of 64 x 64 outputs each for BM = 128, 1 x 4 of 64 x 32 for BM = 64.
// Most calls run in the form whose wavefronts own columns (kq_mm_own.hip), shorter ones in the few-row one (mm_narrow.h).
// Up to four matrices of one K over the same activations share a launch.
//
// Prefill is exempt from the "row r of a batch == row r alone" rule in the reference too
// (src/ops/invariant.rs:140-168): results agree with the mat-vec path to bf16 rounding of
// the weights and the order of the fp32 sums, not bit for bit.
#include <type_traits>

#include "dmath.h"
#include "kq_mm_own.h"
#include "mm_narrow_host.h"
#include "rt.h"

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
// (a native vector: arrays of HIP's uint4 struct that are stored to LDS through casts are left in scratch memory)
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

constexpr int BN = 128, BK = 128, LDK = BK + 8;

struct MmArgs {
  const uint8_t* qs;
  const uint8_t* scales;
  const uint16_t* dm;
  const bf16_t* x;   // [x_rows, K]
  bf16_t* y;         // [y_rows, O]
  int M, O, K;
  // gathered form: tiles over (expert, row range) of an expert-sorted pair list
  const uint32_t* pair;        // [pairs] expert-sorted pair ids (row of y; row of x is pair / up_div)
  int up_div;                  // top_k for the gate / up projections (x row = token), 1 for down
  const uint32_t* tile_expert; // [tiles]
  const uint32_t* tile_start;  // [tiles] first pair
  const uint32_t* tile_count;  // [tiles] pairs in the tile (<= BM)
  const uint32_t* n_tiles;     // device scalar
  int sub;                     // workgroups a plan tile takes (plan tiles may be taller than the kernel's)
  int vec;                     // rows of y can be stored 16 bytes at a time
  // further matrices of the same kind and K over the same activations (plain form): the
  // workgroups from column block bx0 on belong to segment i
  struct Seg {
    const uint8_t* qs;
    const uint8_t* scales;
    const uint16_t* dm;
    bf16_t* y;
    int O, bx0, kind;
  } seg[3];
  int nseg;
  int kind;  // of the first matrix (read by the kernel instance for matrices of both kinds)
};

// the matrix a workgroup of the plain form works on; returns its column block there
__device__ __forceinline__ int pick_segment(MmArgs& a) {
  int bx = blockIdx.x;
#pragma unroll
  for (int i = 0; i < 3; ++i)
    if (i < a.nseg && (int)blockIdx.x >= a.seg[i].bx0) {
      a.qs = a.seg[i].qs;
      a.scales = a.seg[i].scales;
      a.dm = a.seg[i].dm;
      a.y = a.seg[i].y;
      a.O = a.seg[i].O;
      a.kind = a.seg[i].kind;
      bx = (int)blockIdx.x - a.seg[i].bx0;
    }
  return bx;
}

__device__ __forceinline__ uint32_t pack2(float a, float b) { return dm_f2bf2(a, b); }

// ---- weight slab pieces: loaded as codes into registers (so the loads of the next slab can
// be in flight while the matrix cores work on this one), dequantized on the way into LDS ----
struct BRegsQ4 {
  uint4 q0, q1;
  uint32_t s0, s1, s2, dmw;
};
struct BRegsQ6 {
  uint4 qa, qb, qh;
  uint2 sc;
  uint32_t d;
};

// 64-group `grp` of super-block `ib` of weight row `row`
__device__ __forceinline__ BRegsQ4 load_q4k(const MmArgs& a, int64_t row, int nb, int ib, int grp) {
  const int64_t blk = row * nb + ib;
  BRegsQ4 r;
  const uint4* q = reinterpret_cast<const uint4*>(a.qs + blk * 128 + grp * 32);
  r.q0 = q[0];
  r.q1 = q[1];
  const uint32_t* sc = reinterpret_cast<const uint32_t*>(a.scales + blk * 12);
  r.s0 = sc[0];
  r.s1 = sc[1];
  r.s2 = sc[2];
  r.dmw = *reinterpret_cast<const uint32_t*>(a.dm + blk * 2);
  return r;
}

// 64 weights as bf16 into dst[0..64): d*sc*q - dmin*m (kquant::dequantize, q4k.metal:64-96).
// Two and a half vector instructions a weight (byte -> float, one fma, half a two-value bf16
// conversion): the dequantization shares the wavefront with the MFMAs it feeds, so its length
// is GEMM time.
__device__ __forceinline__ void dequant_q4k(const BRegsQ4& r, int grp, bf16_t* dst) {
  // the 6-bit scale and min of sub-blocks 2*grp and 2*grp + 1, two bytes each way
  const int sh16 = (grp & 1) * 16;
  const uint32_t a = r.s0 >> sh16, b = r.s1 >> sh16, c = r.s2 >> sh16;
  const bool low = grp < 2;
  const uint32_t sc16 = low ? (a & 0x3f3fu) : ((c & 0x0f0fu) | ((a & 0xc0c0u) >> 2));
  const uint32_t m16 = low ? (b & 0x3f3fu) : (((c >> 4) & 0x0f0fu) | ((b & 0xc0c0u) >> 2));
  const float d = dm_h2f((f16_t)(r.dmw & 0xffffu)), dmin = dm_h2f((f16_t)(r.dmw >> 16));
  const float dd0 = d * dm_ubyte<0>(sc16), dd1 = d * dm_ubyte<1>(sc16);
  const float mm0 = -(dmin * dm_ubyte<0>(m16)), mm1 = -(dmin * dm_ubyte<1>(m16));
  uint32_t* out = reinterpret_cast<uint32_t*>(dst);
  const uint32_t w[8] = {r.q0.x, r.q0.y, r.q0.z, r.q0.w, r.q1.x, r.q1.y, r.q1.z, r.q1.w};
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const uint32_t lo = w[i] & 0x0f0f0f0fu, hi = (w[i] >> 4) & 0x0f0f0f0fu;
    out[2 * i] = pack2(dm_fma(dd0, dm_ubyte<0>(lo), mm0), dm_fma(dd0, dm_ubyte<1>(lo), mm0));  // low nibbles: weights 4i .. 4i+3
    out[2 * i + 1] = pack2(dm_fma(dd0, dm_ubyte<2>(lo), mm0), dm_fma(dd0, dm_ubyte<3>(lo), mm0));
    out[16 + 2 * i] = pack2(dm_fma(dd1, dm_ubyte<0>(hi), mm1), dm_fma(dd1, dm_ubyte<1>(hi), mm1));  // high nibbles: the same + 32
    out[16 + 2 * i + 1] = pack2(dm_fma(dd1, dm_ubyte<2>(hi), mm1), dm_fma(dd1, dm_ubyte<3>(hi), mm1));
  }
}

// positions l in [16*j, 16*j + 16) of the 128-half `hh` of super-block `ib`
__device__ __forceinline__ BRegsQ6 load_q6k(const MmArgs& a, int64_t row, int nb, int ib, int hh, int j) {
  const int64_t blk = row * nb + ib;
  const uint8_t* base = a.qs + blk * 192;
  BRegsQ6 r;
  r.qa = *reinterpret_cast<const uint4*>(base + 64 * hh + 16 * j);
  r.qb = *reinterpret_cast<const uint4*>(base + 64 * hh + 32 + 16 * j);
  r.qh = *reinterpret_cast<const uint4*>(base + 128 + 32 * hh + 16 * j);
  r.sc = *reinterpret_cast<const uint2*>(a.scales + blk * 16 + 8 * hh);
  r.d = a.dm[blk];
  return r;
}

// the four weights l, l+32, l+64, l+96 of each position, d*sc*(q - 32) (q6k.metal:47-77), as
// bf16 into dst[0..128) (dst = start of the half). The 6-bit codes are put together four at a
// time in a word; (q - 32) * s is one fma with -32 s.
__device__ __forceinline__ void dequant_q6k(const BRegsQ6& r, int j, bf16_t* dst) {
  const float d = dm_h2f((f16_t)r.d);
  const uint32_t scw[2] = {r.sc.x, r.sc.y};
  auto scale = [&](int i) { return (float)(int)(int8_t)((scw[i >> 2] >> (8 * (i & 3))) & 0xffu); };
  const float sv[4] = {d * scale(j), d * scale(j + 2), d * scale(j + 4), d * scale(j + 6)};
  const float off[4] = {-32.f * sv[0], -32.f * sv[1], -32.f * sv[2], -32.f * sv[3]};
  const uint32_t la[4] = {r.qa.x, r.qa.y, r.qa.z, r.qa.w}, lb[4] = {r.qb.x, r.qb.y, r.qb.z, r.qb.w},
                 hv[4] = {r.qh.x, r.qh.y, r.qh.z, r.qh.w};
  uint32_t* out = reinterpret_cast<uint32_t*>(dst);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t A = la[i], B = lb[i], H = hv[i];
    const uint32_t c[4] = {(A & 0x0f0f0f0fu) | ((H << 4) & 0x30303030u), (B & 0x0f0f0f0fu) | ((H << 2) & 0x30303030u),
                           ((A >> 4) & 0x0f0f0f0fu) | (H & 0x30303030u), ((B >> 4) & 0x0f0f0f0fu) | ((H >> 2) & 0x30303030u)};
    const int e = (16 * j + 4 * i) >> 1;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      out[16 * g + e] = pack2(dm_fma(sv[g], dm_ubyte<0>(c[g]), off[g]), dm_fma(sv[g], dm_ubyte<1>(c[g]), off[g]));
      out[16 * g + e + 1] = pack2(dm_fma(sv[g], dm_ubyte<2>(c[g]), off[g]), dm_fma(sv[g], dm_ubyte<3>(c[g]), off[g]));
    }
  }
}

template <int KIND>
struct BRegsOf { typedef BRegsQ4 type; };
template <>
struct BRegsOf<ORNITH_Q6K> { typedef BRegsQ6 type; };

// ---- epilogue ------------------------------------------------------------------------------
// The MFMA result has one output column per lane (D[row = 8*b + 4*(lane/32) + r][col = lane%32]
// = acc[4*b + r]): stored from there, a tile row leaves in 2-byte pieces, 64 store instructions
// per 32 x 32 tile. Each wavefront instead turns its own window of the tile around in LDS (the
// slab buffers are free after the last barrier; no other wavefront touches the window, so no
// barrier is needed) and stores 16 bytes a lane, eight lanes a 128-byte row piece. `vec`: the
// rows of y are 16-byte aligned (O a multiple of 8); otherwise the direct 2-byte stores.
template <int TM, int TN, bool GATHER>
__device__ __forceinline__ void store_tile(const MmArgs& a, const f32x16_t (&acc)[TM][TN], bf16_t* cs, int row0,
                                           int col0, int lane, int n0, int m0, int rows_here, const uint32_t* s_dst,
                                           bool vec, int ld = LDK) {
  constexpr int WTM = TM * 32, WTN = TN * 32, PPR = WTN / 8;
  if (!vec) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int o = n0 + col0 + j * 32 + (lane & 31);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int r = row0 + i * 32 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
          if (r < rows_here && o < a.O) {
            const int64_t dst = GATHER ? (int64_t)s_dst[r] : (int64_t)(m0 + r);
            a.y[dst * a.O + o] = dm_f2bf(acc[i][j][e]);
          }
        }
      }
    return;
  }
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      bf16_t* w = cs + (row0 + i * 32 + 4 * (lane >> 5)) * ld + col0 + j * 32 + (lane & 31);
#pragma unroll
      for (int e = 0; e < 16; e += 2) {
        const uint32_t pk = dm_f2bf2(acc[i][j][e], acc[i][j][e + 1]);
        w[(8 * (e >> 2) + (e & 3)) * ld] = (bf16_t)(pk & 0xffffu);
        w[(8 * (e >> 2) + (e & 3) + 1) * ld] = (bf16_t)(pk >> 16);
      }
    }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
  for (int p0 = 0; p0 < WTM * PPR; p0 += 64) {
    const int p = p0 + lane, r = row0 + p / PPR, c = col0 + (p % PPR) * 8;
    if (r < rows_here && n0 + c < a.O) {
      const int64_t dst = GATHER ? (int64_t)s_dst[r] : (int64_t)(m0 + r);
      *reinterpret_cast<u32x4_t*>(a.y + dst * a.O + n0 + c) = *reinterpret_cast<const u32x4_t*>(cs + r * ld + c);
    }
  }
}

// BM = 128: 2 x 2 wavefronts of 64 x 64; BM = 64: 1 x 4 of 64 x 32; BM = 256: 2 x 2 of 128 x 64 (plain, enough tiles to fill the device: matrices
// or activations that are not 16-byte aligned or past 32-bit offsets, and gemm_duo = 0).
// KIND = kMixed: the matrices of the launch differ in kind (a workgroup asks its own).
constexpr int kMixed = 2;
template <int KIND, int BM, bool GATHER>
__global__ __launch_bounds__(256) void kq_mm_kernel(MmArgs a) {
  constexpr int WM = BM >= 128 ? 2 : 1, WN = 4 / WM;
  constexpr int WTM = BM / WM, WTN = BN / WN;
  constexpr int TM = WTM / 32, TN = WTN / 32;
  constexpr int NA = BM * 16 / 256;  // 16-byte pieces of the activation slab per thread
  __shared__ __attribute__((aligned(16))) bf16_t As[BM][LDK];
  __shared__ __attribute__((aligned(16))) bf16_t Bs[BN][LDK];
  __shared__ uint32_t s_src[BM], s_dst[BM];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WN, wn = wave % WN;
  const int n0 = (GATHER ? (int)blockIdx.x : pick_segment(a)) * BN;
  const int nb = a.K >> 8;

  int rows_here, m0 = 0;
  int64_t wrow0 = 0;  // first weight row of this tile's matrix
  if constexpr (GATHER) {
    // a plan tile of more rows than BM is worked on by a.sub workgroups, BM rows each
    const uint32_t tile = blockIdx.y / (uint32_t)a.sub, part = blockIdx.y % (uint32_t)a.sub;
    if (tile >= *a.n_tiles) return;
    const uint32_t e = a.tile_expert[tile], st = a.tile_start[tile] + part * BM;
    rows_here = min((int)a.tile_count[tile] - (int)(part * BM), BM);
    if (rows_here <= 0) return;
    wrow0 = (int64_t)e * a.O;
    for (int r = tid; r < BM; r += 256) {
      const uint32_t p = r < rows_here ? a.pair[st + r] : 0u;
      s_src[r] = p / (uint32_t)a.up_div;
      s_dst[r] = p;
    }
    __syncthreads();
  } else {
    m0 = blockIdx.y * BM;
    rows_here = min(BM, a.M - m0);
  }

  // this thread's pieces of a slab: NA activation pieces and one weight piece
  const int br = tid >> 1, bpart = tid & 1;
  const int64_t brow = wrow0 + min(n0 + br, a.O - 1);
  const bf16_t* asrc[NA];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int idx = tid + 256 * i, r = idx >> 4, c8 = idx & 15;
    // rows past the end of the tile read a valid row instead (pair 0's, or the last one): what
    // they produce lands in output rows the epilogue does not store, and no load needs a branch
    const int64_t src = GATHER ? (int64_t)s_src[r] : (int64_t)min(m0 + r, a.M - 1);
    asrc[i] = a.x + src * a.K + 8 * c8;
  }
  u32x4_t areg[NA];
  BRegsQ4 breg4;
  BRegsQ6 breg6;
  const bool q4 = KIND == kMixed ? a.kind == ORNITH_Q4K : KIND == ORNITH_Q4K;
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < NA; ++i)
      areg[i] = *reinterpret_cast<const u32x4_t*>(asrc[i] + k0);
    if (q4)
      breg4 = load_q4k(a, brow, nb, k0 >> 8, ((k0 & 255) >> 6) + bpart);
    else
      breg6 = load_q6k(a, brow, nb, k0 >> 8, (k0 & 255) >> 7, bpart);
  };

  f32x16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  fetch(0);
  for (int k0 = 0; k0 < a.K; k0 += BK) {
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      const int idx = tid + 256 * i;
      *reinterpret_cast<u32x4_t*>(&As[idx >> 4][8 * (idx & 15)]) = areg[i];
    }
    if (q4)
      dequant_q4k(breg4, ((k0 & 255) >> 6) + bpart, &Bs[br][64 * bpart]);
    else
      dequant_q6k(breg6, bpart, &Bs[br][0]);
    __syncthreads();
    if (k0 + BK < a.K) fetch(k0 + BK);  // in flight while the matrix cores run
    // fragments of step kk + 1 leave LDS while the matrix cores work on step kk
    bf16x8_t af[2][TM], bfr[2][TN];
    auto frags = [&](int kk, bf16x8_t (&fa)[TM], bf16x8_t (&fb)[TN]) {
      const int kc = kk * 16 + 8 * (lane >> 5);
#pragma unroll
      for (int i = 0; i < TM; ++i)
        fa[i] = *reinterpret_cast<const bf16x8_t*>(&As[wm * WTM + i * 32 + (lane & 31)][kc]);
#pragma unroll
      for (int j = 0; j < TN; ++j)
        fb[j] = *reinterpret_cast<const bf16x8_t*>(&Bs[wn * WTN + j * 32 + (lane & 31)][kc]);
    };
    frags(0, af[0], bfr[0]);
#pragma unroll
    for (int kk = 0; kk < BK / 16; ++kk) {
      if (kk + 1 < BK / 16) frags(kk + 1, af[(kk + 1) & 1], bfr[(kk + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);  // or the reads are sunk to just before their use
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[kk & 1][i], bfr[kk & 1][j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }

  store_tile<TM, TN, GATHER>(a, acc, &As[0][0], wm * WTM, wn * WTN, lane, n0, m0, rows_here, s_dst, a.vec != 0);
}

// BM == 64 has two 32-row MFMA tiles per wavefront as well (TM = 2), one wavefront column
static_assert(BN == 128 && BK == 128, "tile constants are baked into the index arithmetic");

// ---- expert-sorted pair list for the gathered form -----------------------------------
// inds [pairs] (expert of pair p; pair p = token * k + slot). One workgroup: counts per expert,
// exclusive scan, scatter, then the tile list, fullest tiles first (the GEMM's workgroups start
// in the order of the list, and one that starts late with many rows would be the tail).
constexpr int kSortTilesMax = 2048;  // tile lists up to this length are ordered

// Writes the tile list fullest first: a counting sort over the tile heights (a tile has 1 .. bm
// <= 256 rows; tiles of one height land in the order their atomics are served, which changes
// the order workgroups start in and nothing else). All 1024 threads of the workgroup call it.
__device__ __forceinline__ void order_tiles(uint32_t total_tiles, int bm, const uint32_t* t_expert, const uint32_t* t_start,
                                            const uint32_t* t_count, uint32_t* tile_expert, uint32_t* tile_start,
                                            uint32_t* tile_count) {
  __shared__ uint32_t bin[257];
  const int tid = threadIdx.x;
  if (tid < 257) bin[tid] = 0;
  __syncthreads();
  for (uint32_t i = tid; i < total_tiles; i += 1024) atomicAdd(&bin[min(t_count[i], 256u)], 1u);
  __syncthreads();
  if (tid == 0) {  // places of the heights, tallest first
    uint32_t at = 0;
    for (int c = min(bm, 256); c >= 0; --c) {
      const uint32_t n = bin[c];
      bin[c] = at;
      at += n;
    }
  }
  __syncthreads();
  for (uint32_t i = tid; i < total_tiles; i += 1024) {
    const uint32_t c = t_count[i], at = atomicAdd(&bin[min(c, 256u)], 1u);
    tile_expert[at] = t_expert[i];
    tile_start[at] = t_start[i];
    tile_count[at] = c;
  }
}


// The tiles of the shared expert, which every token goes through: number E, "pairs" pairs + t. They
// follow the routed ones in the list. Returns how many there are.
__device__ __forceinline__ uint32_t shared_tiles(int shared_rows, int pairs, int E, int bm, uint32_t at, uint32_t* t_expert,
                                                 uint32_t* t_start, uint32_t* t_count, uint32_t* pair) {
  const uint32_t n = (uint32_t)(shared_rows + bm - 1) / bm;
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
    t_expert[at + i] = E;
    t_start[at + i] = pairs + i * bm;
    t_count[at + i] = min((uint32_t)bm, (uint32_t)shared_rows - i * bm);
  }
  for (int i = threadIdx.x; i < shared_rows; i += blockDim.x) pair[pairs + i] = pairs + i;
  return n;
}

__global__ __launch_bounds__(1024) void moe_sort_pairs_kernel(const uint32_t* inds, int pairs, int E,
                                                              int bm, int shared_rows, uint32_t* pair, uint32_t* tile_expert,
                                                              uint32_t* tile_start, uint32_t* tile_count,
                                                              uint32_t* n_tiles, uint32_t* expert_at) {
  __shared__ uint32_t cnt[1024], fill[1024];
  __shared__ unsigned long long scan[2][1024];  // pairs before an expert (low 40 bits) and tiles before it
  __shared__ uint32_t t_expert[kSortTilesMax], t_start[kSortTilesMax], t_count[kSortTilesMax];
  const int tid = threadIdx.x;
  cnt[tid] = 0;
  fill[tid] = 0;
  __syncthreads();
  // (eight loads in flight a thread: one after the other, each pass over the pairs is 32 memory
  // latencies long for a 4096-token chunk)
  for (int p0 = tid; p0 < pairs; p0 += 8 * 1024) {
    uint32_t e[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) e[u] = p0 + 1024 * u < pairs ? inds[p0 + 1024 * u] : 0u;
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (p0 + 1024 * u < pairs) atomicAdd(&cnt[min(e[u], (uint32_t)(E - 1))], 1u);
  }
  __syncthreads();
  // inclusive scan over the 1024 slots (experts past E hold zero), ten doubling steps
  const uint32_t mine = cnt[tid];
  scan[0][tid] = (unsigned long long)mine | ((unsigned long long)((mine + bm - 1) / bm) << 40);
  __syncthreads();
  int cur = 0;
  for (int d = 1; d < 1024; d <<= 1) {
    const unsigned long long v = scan[cur][tid] + (tid >= d ? scan[cur][tid - d] : 0ull);
    scan[cur ^ 1][tid] = v;
    cur ^= 1;
    __syncthreads();
  }
  const unsigned long long incl = scan[cur][tid];
  const uint32_t my_tiles = (mine + bm - 1) / bm;
  const uint32_t start = (uint32_t)(incl & ((1ull << 40) - 1)) - mine;
  const uint32_t tiles_before = (uint32_t)(incl >> 40) - my_tiles;
  const uint32_t routed_tiles = (uint32_t)(scan[cur][1023] >> 40);
  const uint32_t total_tiles = routed_tiles + (uint32_t)(shared_rows + bm - 1) / bm;
  if (tid == 0) *n_tiles = total_tiles;
  __syncthreads();
  scan[0][tid] = start;  // (reused: where an expert's run of pairs begins)
  if (tid < E) expert_at[tid] = start;
  __syncthreads();
  // placement: a pair takes the next free place of its expert. The order inside an expert's
  // run depends on the scheduling of the atomics, the results do not: every output row is one
  // dot product over k in a fixed order, whichever tile row computes it.
  for (int p0 = tid; p0 < pairs; p0 += 8 * 1024) {
    uint32_t e[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) e[u] = p0 + 1024 * u < pairs ? min(inds[p0 + 1024 * u], (uint32_t)(E - 1)) : 0u;
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (p0 + 1024 * u < pairs) pair[(uint32_t)scan[0][e[u]] + atomicAdd(&fill[e[u]], 1u)] = (uint32_t)(p0 + 1024 * u);
  }
  const bool ordered = total_tiles <= (uint32_t)kSortTilesMax;
  if (tid < E)
    for (uint32_t t = 0; t < my_tiles; ++t) {
      const uint32_t i = tiles_before + t, st = start + t * bm, c = min((uint32_t)bm, mine - t * bm);
      if (ordered) {
        t_expert[i] = tid;
        t_start[i] = st;
        t_count[i] = c;
      } else {
        tile_expert[i] = tid;
        tile_start[i] = st;
        tile_count[i] = c;
      }
    }
  if (ordered) shared_tiles(shared_rows, pairs, E, bm, routed_tiles, t_expert, t_start, t_count, pair);
  else shared_tiles(shared_rows, pairs, E, bm, routed_tiles, tile_expert, tile_start, tile_count, pair);
  __syncthreads();
  if (!ordered) return;
  order_tiles(total_tiles, bm, t_expert, t_start, t_count, tile_expert, tile_start, tile_count);
}

// ---- the same plan from many workgroups -----------------------------------------------
// A pass over the pairs is one LDS atomic a pair, about a cycle each in one workgroup: 33 us
// for the 32768 pairs of a 4096-token chunk. From 8192 pairs on, kSortParts workgroups count
// their slices of the pairs side by side, one workgroup turns the counts into places (per
// expert, then per slice inside an expert's run) and writes the tile list, and the slices
// scatter side by side.
constexpr int kSortParts = 32;

__global__ __launch_bounds__(256) void moe_sort_count_kernel(const uint32_t* inds, int pairs, int E, uint32_t* part_cnt) {
  __shared__ uint32_t cnt[1024];
  for (int e = threadIdx.x; e < E; e += 256) cnt[e] = 0;
  __syncthreads();
  const int per = (pairs + kSortParts - 1) / kSortParts, a = blockIdx.x * per, b = min(pairs, a + per);
  for (int p = a + threadIdx.x; p < b; p += 256) atomicAdd(&cnt[min(inds[p], (uint32_t)(E - 1))], 1u);
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += 256) part_cnt[blockIdx.x * E + e] = cnt[e];
}

// part_cnt [parts, E] in: pairs of expert e in slice b; out: where slice b's pairs of expert e begin (slice 0: the expert's)
__global__ __launch_bounds__(1024) void moe_sort_plan_kernel(int pairs, int E, int bm, int shared_rows, uint32_t* part_cnt,
                                                             uint32_t* pair, uint32_t* tile_expert,
                                                             uint32_t* tile_start, uint32_t* tile_count,
                                                             uint32_t* n_tiles) {
  __shared__ unsigned long long scan[2][1024];
  __shared__ uint32_t t_expert[kSortTilesMax], t_start[kSortTilesMax], t_count[kSortTilesMax];
  const int tid = threadIdx.x;
  uint32_t mine = 0;
  if (tid < E)
    for (int b = 0; b < kSortParts; ++b) mine += part_cnt[b * E + tid];
  const uint32_t my_tiles = (mine + bm - 1) / bm;
  scan[0][tid] = (unsigned long long)mine | ((unsigned long long)my_tiles << 40);
  __syncthreads();
  int cur = 0;
  for (int d = 1; d < 1024; d <<= 1) {
    const unsigned long long v = scan[cur][tid] + (tid >= d ? scan[cur][tid - d] : 0ull);
    scan[cur ^ 1][tid] = v;
    cur ^= 1;
    __syncthreads();
  }
  const unsigned long long incl = scan[cur][tid];
  const uint32_t start = (uint32_t)(incl & ((1ull << 40) - 1)) - mine;
  const uint32_t tiles_before = (uint32_t)(incl >> 40) - my_tiles;
  const uint32_t routed_tiles = (uint32_t)(scan[cur][1023] >> 40);
  const uint32_t total_tiles = routed_tiles + (uint32_t)(shared_rows + bm - 1) / bm;
  if (tid == 0) *n_tiles = total_tiles;
  if (tid < E) {
    uint32_t at = start;
    for (int b = 0; b < kSortParts; ++b) {
      const uint32_t c = part_cnt[b * E + tid];
      part_cnt[b * E + tid] = at;
      at += c;
    }
  }
  const bool ordered = total_tiles <= (uint32_t)kSortTilesMax;
  if (tid < E)
    for (uint32_t t = 0; t < my_tiles; ++t) {
      const uint32_t i = tiles_before + t, st = start + t * bm, c = min((uint32_t)bm, mine - t * bm);
      if (ordered) {
        t_expert[i] = tid;
        t_start[i] = st;
        t_count[i] = c;
      } else {
        tile_expert[i] = tid;
        tile_start[i] = st;
        tile_count[i] = c;
      }
    }
  if (ordered) shared_tiles(shared_rows, pairs, E, bm, routed_tiles, t_expert, t_start, t_count, pair);
  else shared_tiles(shared_rows, pairs, E, bm, routed_tiles, tile_expert, tile_start, tile_count, pair);
  __syncthreads();
  if (!ordered) return;
  order_tiles(total_tiles, bm, t_expert, t_start, t_count, tile_expert, tile_start, tile_count);
}

__global__ __launch_bounds__(256) void moe_sort_scatter_kernel(const uint32_t* inds, int pairs, int E,
                                                               const uint32_t* part_at, uint32_t* pair) {
  __shared__ uint32_t at[1024];
  for (int e = threadIdx.x; e < E; e += 256) at[e] = part_at[blockIdx.x * E + e];
  __syncthreads();
  const int per = (pairs + kSortParts - 1) / kSortParts, a = blockIdx.x * per, b = min(pairs, a + per);
  for (int p = a + threadIdx.x; p < b; p += 256) pair[atomicAdd(&at[min(inds[p], (uint32_t)(E - 1))], 1u)] = (uint32_t)p;
}

int check(const ornith_kmatrix* w, const char* who) {
  ORN_REQUIRE(w && (w->kind == ORNITH_Q4K || w->kind == ORNITH_Q6K), "%s: bad matrix", who);
  ORN_REQUIRE(w->K >= 256 && w->K % 256 == 0 && w->O >= 1 && w->E >= 1, "%s: bad dims E=%d O=%d K=%d", who,
              w->E, w->O, w->K);
  ORN_REQUIRE(w->d_qs && w->d_scales && w->d_dm, "%s: null tensor", who);
  return ORNITH_OK;
}

}  // namespace

// What a plan takes: pairs and tile list of the routed experts and, if shared_rows > 0, of the shared one.
size_t moe_plan_bytes(int pairs, int E, int rows, int shared_rows) {
  const size_t tiles = (size_t)pairs / rows + (size_t)E + 1 + (size_t)(shared_rows + rows - 1) / rows;
  return ((size_t)pairs + shared_rows + tiles * 3 + 1 + (size_t)kSortParts * E) * 4 + 6 * 256;
}

// Lays the plan out in d_plan; with `build` it is made from the pairs' experts first.
int moe_plan(ornith_ctx* ctx, const uint32_t* d_inds, int pairs, int E, int rows, int shared_rows, void* d_plan, bool build,
             nmm::Plan* out) {
  nmm::Plan p{};
  p.rows = rows;
  p.tiles_max = (size_t)pairs / rows + (size_t)E + 1 + (size_t)(shared_rows + rows - 1) / rows;
  ScratchCursor pc(d_plan);
  p.pair = pc.take<uint32_t>((size_t)pairs + shared_rows);
  p.tile_expert = pc.take<uint32_t>(p.tiles_max);
  p.tile_start = pc.take<uint32_t>(p.tiles_max);
  p.tile_count = pc.take<uint32_t>(p.tiles_max);
  p.n_tiles = pc.take<uint32_t>(1);
  uint32_t* parts = pc.take<uint32_t>((size_t)kSortParts * E);
  p.expert_at = parts;
  if (build && pairs >= 8192) {
    hipLaunchKernelGGL(moe_sort_count_kernel, dim3(kSortParts), dim3(256), 0, ctx->stream, d_inds, pairs, E, parts);
    hipLaunchKernelGGL(moe_sort_plan_kernel, dim3(1), dim3(1024), 0, ctx->stream, pairs, E, rows, shared_rows, parts, p.pair,
                       p.tile_expert, p.tile_start, p.tile_count, p.n_tiles);
    hipLaunchKernelGGL(moe_sort_scatter_kernel, dim3(kSortParts), dim3(256), 0, ctx->stream, d_inds, pairs, E, parts, p.pair);
    ORN_LAUNCH_CHECK("moe_sort_*_kernel");
  } else if (build) {
    hipLaunchKernelGGL(moe_sort_pairs_kernel, dim3(1), dim3(1024), 0, ctx->stream, d_inds, pairs, E, rows, shared_rows,
                       p.pair, p.tile_expert, p.tile_start, p.tile_count, p.n_tiles, parts);
    ORN_LAUNCH_CHECK("moe_sort_pairs_kernel");
  }
  *out = p;
  return ORNITH_OK;
}

extern "C" {

// Up to four matrices of one K over the same activations (the projections that share an input: narrow ones alone
// leave compute units without a workgroup). Those that suit the form whose wavefronts own columns share a launch of
// it; of the others those of one kind take the tile the whole launch's size calls for, a mix of kinds 128-row tiles.
int ornith_kq_matmul_multi(ornith_ctx* ctx, const ornith_kmatrix* const* ws, int n, const void* d_x, int M,
                           void* const* d_ys) {
  ORN_REQUIRE(ctx && ws && d_x && d_ys && n >= 1 && n <= 4, "kq_matmul: bad argument");
  ORN_REQUIRE(M >= 1, "kq_matmul: M=%d", M);
  ORN_REQUIRE(((uintptr_t)d_x & 15) == 0, "kq_matmul: x must be 16-byte aligned");
  MmArgs a{};
  OwnArgs own[2] = {};  // those that take halves of K go by themselves
  int nx = 0, rest = 0;
  bool mixed = false;
  a.vec = 1;
  for (int i = 0; i < n; ++i) {
    ORN_REQUIRE(ws[i] && d_ys[i], "kq_matmul: null entry %d", i);
    int rc = check(ws[i], "kq_matmul");
    if (rc) return rc;
    ORN_REQUIRE(ws[i]->E == 1, "kq_matmul: stacked matrix (use kq_gather_matmul)");
    ORN_REQUIRE(ws[i]->K == ws[0]->K, "kq_matmul: matrices of one launch differ in K");
  }
  for (int i = 0; i < n; ++i) {
    if (kq_mm_own_suits(*ws[i], d_x, M)) {
      OwnArgs& o = own[kq_mm_own_halves(*ws[i], M)];
      o.m[o.n++] = kq_mm_own_mat(*ws[i], d_ys[i]);
      continue;
    }
    a.vec = a.vec && ws[i]->O % 8 == 0 && ((uintptr_t)d_ys[i] & 15) == 0;
    if (rest == 0) {
      a.qs = (const uint8_t*)ws[i]->d_qs;
      a.scales = (const uint8_t*)ws[i]->d_scales;
      a.dm = (const uint16_t*)ws[i]->d_dm;
      a.y = (bf16_t*)d_ys[i];
      a.O = ws[i]->O;
      a.kind = ws[i]->kind;
    } else {
      a.seg[rest - 1] = {(const uint8_t*)ws[i]->d_qs, (const uint8_t*)ws[i]->d_scales, (const uint16_t*)ws[i]->d_dm,
                         (bf16_t*)d_ys[i], ws[i]->O, nx, ws[i]->kind};
    }
    mixed = mixed || ws[i]->kind != a.kind;
    nx += (ws[i]->O + BN - 1) / BN;
    ++rest;
  }
  for (const bool halves : {false, true}) {
    OwnArgs& o = own[halves];
    if (!o.n) continue;
    o.x = (const bf16_t*)d_x;
    o.M = M;
    o.K = ws[0]->K;
    o.halves = halves;
    if (const int rc = kq_mm_own(ctx, o, false)) return rc;
  }
  if (!rest) return ORNITH_OK;
  a.nseg = rest - 1;
  a.x = (const bf16_t*)d_x;
  a.M = M;
  a.K = ws[0]->K;
  // 256-row tiles dequantize every weight tile half as often; 128-row tiles when that is what
  // it takes to give every compute unit a workgroup
  const bool big = !mixed && M >= 256 && (long)nx * ((M + 255) / 256) >= ctx->compute_units;
  const dim3 grid(nx, big ? (M + 255) / 256 : (M + 127) / 128);
  typedef void (*Kernel)(MmArgs);
  const Kernel k = mixed ? kq_mm_kernel<kMixed, 128, false>
                   : a.kind == ORNITH_Q4K ? (big ? kq_mm_kernel<ORNITH_Q4K, 256, false> : kq_mm_kernel<ORNITH_Q4K, 128, false>)
                                          : (big ? kq_mm_kernel<ORNITH_Q6K, 256, false> : kq_mm_kernel<ORNITH_Q6K, 128, false>);
  hipLaunchKernelGGL(k, grid, dim3(256), 0, ctx->stream, a);
  ORN_LAUNCH_CHECK("kq_mm_kernel");
  return ORNITH_OK;
}

int ornith_kq_matmul(ornith_ctx* ctx, const ornith_kmatrix* w, const void* d_x, int M, void* d_y) {
  ORN_REQUIRE(w && d_y, "kq_matmul: null argument");
  return ornith_kq_matmul_multi(ctx, &w, 1, d_x, M, &d_y);
}

}  // extern "C"

namespace {

// Pairs an expert from which a matrix that the few-row kernels don't take runs in the form whose wavefronts own columns, for K >= 1024 (us, LDS form / there, Q4_K, 48 rows an
// expert: 512 x 4352, 4 / 64 / 128 experts 42 / 29, 67 / 48, 108 / 97, 2048 x 8192, 8 experts 93 / 61; fewer slabs, 2048 x 256 at 16 / 256
// experts 6.6 / 7.6, 50 / 56, 131 x 512 at 16 / 256 8.9 / 10, 17 / 19).
constexpr int kOwnPairs = 48;

struct GatherRoute {
  int tile_rows;  // of the plan: depends only on pairs and E (and the option), so the calls sharing a plan agree on it
  int lds_rows;   // a workgroup's in the LDS form
  bool few, own, low;
};

// Rows per plan tile: with nmm::kNarrowPairs rows an expert or more 256, the own-column form's most: nearly every expert
// is one tile there (its weights are dequantized once), and one of fewer rows runs the loop for the rows it has.
// Otherwise the few-row kernels' 16 / 32 / 64 rows, the smallest that most experts' shares fit.
// The kernel for this matrix: with few rows an expert the few-row kernels (mm_narrow.h). Tall plans, and from kOwnPairs rows an
// expert on the matrices that the few-row kernels don't take (K > 4096, rows whose scales are no whole 16-byte
// pieces; their 64-row tiles are worked on four at a time), take the own-column form where its alignment holds.
// Otherwise the LDS form: 128 rows a workgroup from 96 rows an expert on and K >= 1024, else 64. A plan tile
// taller than its kernel's workgroups is split over several of them.
GatherRoute gather_route(const ornith_kmatrix& w, const void* d_x, int pairs, int top_k, bool is_up, const void* d_y) {
  const int avg = pairs / w.E;
  const bool narrow = pairs < nmm::kNarrowPairs * w.E, reg = ornith_option_gemm_reg();
  const size_t x_rows = (size_t)(is_up ? pairs / top_k : pairs);
  GatherRoute r;
  r.tile_rows = narrow ? nmm::tile_rows(pairs, w.E) : reg ? kOwnRows : avg >= 96 ? 128 : 64;
  r.lds_rows = avg >= 96 && w.K >= 1024 ? 128 : 64;
  r.few = narrow && nmm::experts_ok(&w, d_x, x_rows, d_y);
  r.low = narrow && !r.few && pairs >= kOwnPairs * w.E && w.K >= 1024 && reg;
  r.own = ((reg && !narrow) || r.low) && kq_mm_own_ok(w, d_x, x_rows);
  return r;
}

}  // namespace

int kq_gather_form(const ornith_kmatrix& w, const void* d_x, int pairs, int top_k, bool is_up, const void* d_y, int units) {
  const GatherRoute r = gather_route(w, d_x, pairs, top_k, is_up, d_y);
  return r.few ? 3 : !r.own ? 0 : kq_mm_own_thin_experts(w.O, w.E, pairs, units) ? 4 : 1;
}

extern "C" {

// gather plan: expert-sorted pairs and the tile list, in caller-provided device memory
// (ornith_kq_gather_plan_bytes(pairs, E) bytes)
size_t ornith_kq_gather_plan_bytes(int pairs, int E) { return moe_plan_bytes(pairs, E, 16, 0); }

int ornith_kq_gather_matmul(ornith_ctx* ctx, const ornith_kmatrix* w, const void* d_x,
                            const uint32_t* d_inds, int pairs, int top_k, int is_up, void* d_plan,
                            int rebuild_plan, void* d_y) {
  ORN_REQUIRE(ctx && d_x && d_inds && d_plan && d_y, "kq_gather_matmul: null argument");
  int rc = check(w, "kq_gather_matmul");
  if (rc) return rc;
  ORN_REQUIRE(pairs >= 1 && top_k >= 1 && pairs % top_k == 0 && w->E <= 1024,
              "kq_gather_matmul: pairs=%d top_k=%d E=%d", pairs, top_k, w->E);
  const GatherRoute r = gather_route(*w, d_x, pairs, top_k, is_up != 0, d_y);
  nmm::Plan pl;
  rc = moe_plan(ctx, d_inds, pairs, w->E, r.tile_rows, 0, d_plan, rebuild_plan != 0, &pl);
  if (rc) return rc;
  if (r.few) return nmm::gathered(ctx, w, nullptr, d_x, pairs, is_up ? top_k : 1, pl, d_y);
  if (r.own) {
    OwnArgs o{};
    o.m[0] = kq_mm_own_mat(*w, d_y);
    o.n = 1;
    o.x = (const bf16_t*)d_x;
    o.M = pairs;
    o.K = w->K;
    o.pair = pl.pair;
    o.tile_expert = pl.tile_expert;
    o.tile_start = pl.tile_start;
    o.tile_count = pl.tile_count;
    o.n_tiles = pl.n_tiles;
    o.tiles_max = (int)pl.tiles_max;
    o.up_div = is_up ? top_k : 1;
    o.expert_at = r.low ? pl.expert_at : nullptr;
    o.E = w->E;
    return kq_mm_own(ctx, o, true);
  }
  MmArgs a{};
  a.qs = (const uint8_t*)w->d_qs;
  a.scales = (const uint8_t*)w->d_scales;
  a.dm = (const uint16_t*)w->d_dm;
  a.x = (const bf16_t*)d_x;
  a.y = (bf16_t*)d_y;
  a.M = pairs;
  a.O = w->O;
  a.K = w->K;
  a.vec = w->O % 8 == 0 && ((uintptr_t)d_y & 15) == 0;
  a.pair = pl.pair;
  a.up_div = is_up ? top_k : 1;
  a.tile_expert = pl.tile_expert;
  a.tile_start = pl.tile_start;
  a.tile_count = pl.tile_count;
  a.n_tiles = pl.n_tiles;
  a.sub = (r.tile_rows + r.lds_rows - 1) / r.lds_rows;
  const dim3 grid((w->O + BN - 1) / BN, (unsigned)(pl.tiles_max * a.sub));
  if (r.lds_rows == 128) {
    if (w->kind == ORNITH_Q4K)
      hipLaunchKernelGGL((kq_mm_kernel<ORNITH_Q4K, 128, true>), grid, dim3(256), 0, ctx->stream, a);
    else
      hipLaunchKernelGGL((kq_mm_kernel<ORNITH_Q6K, 128, true>), grid, dim3(256), 0, ctx->stream, a);
  } else if (w->kind == ORNITH_Q4K)
    hipLaunchKernelGGL((kq_mm_kernel<ORNITH_Q4K, 64, true>), grid, dim3(256), 0, ctx->stream, a);
  else
    hipLaunchKernelGGL((kq_mm_kernel<ORNITH_Q6K, 64, true>), grid, dim3(256), 0, ctx->stream, a);
  ORN_LAUNCH_CHECK("kq_mm_kernel<gather>");
  return ORNITH_OK;
}

}  // extern "C"
