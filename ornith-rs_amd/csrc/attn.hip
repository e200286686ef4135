// Full-attention layer at decode / verify width: per-head RMS + partial RoPE +
// KV append in one kernel, split-K attention over the cache, merge + output gate.
//
// Replaces the middle of Attention::forward
// (/root/reference/src/model/qwen3_5.rs:430-474): rms_norm on q/k heads,
// rope (/root/reference/src/ops/rope.rs:6-60, vendored rope.metal:11-67),
// KvCache::update_and_fetch (/root/reference/src/model/cache.rs:38-79),
// attention_with_cache -> sdpa_vector[_2pass]
// (/root/reference/src/ops/sdpa.rs:33-83,166-264, vendored sdpa_vector.h:15-318)
// and sigmoid_gate (kernels/ornith_elementwise.metal).
//
// Attention is split over keys in blocks of 256 by absolute position, one
// workgroup per (block, query head, query row), or for four or eight heads of a KV group
// where there are many of them: a key's score is one fma chain per
// 64 channels with the chains added pairwise, a channel's output one fma chain per
// 64 keys of the block added the same way, so neither needs a cross-lane reduction
// per key. The partial (max, sum, values) of each block go to scratch and a second
// kernel merges them in ascending block order and applies the sigmoid output gate;
// when every row has a single block the partial kernel does that itself.
// A query row only ever sees keys at or before its own position, and blocks are
// aligned to absolute positions, so row r of a T-row verify call is bit-identical
// to a one-row call at that position.
#include <type_traits>

#include "dmath.h"
#include "rt.h"

namespace {

constexpr int ATT_KB = 256;

struct PrepArgs {
  const bf16_t* qg;  // [T, Hq, 2*hd]
  const bf16_t* kx;  // [T, Hkv, hd]
  const bf16_t* vx;  // [T, Hkv, hd]
  const bf16_t* qw;  // [hd]
  const bf16_t* kw;  // [hd]
  const float* cos_t;  // [npos, half]
  const float* sin_t;
  const int* d_offset;  // optional: position of the first new row, read on the device
  bf16_t* q_rot;      // [T, Hq, hd]
  bf16_t* k_cache;    // [Hkv, cap, hd]
  bf16_t* v_cache;
  int T, Hq, Hkv, offset, cap, npos, half;
  float eps;
};

// The per-head prep of one row by one wavefront (PER = hd / 64 contiguous channels a lane), in
// two steps so that a caller can put other loads between the request and the arithmetic:
// prep_issue asks for the row, the norm weight and the lane's cos / sin entries; prep_finish
// returns the normed, rotated values (rounded to bf16 by whoever stores them).
template <int PER>
struct PrepRegs {
  uint32_t x[PER / 2], w[PER / 2];  // pairs
  float c[PER], s[PER];
};

template <int PER, bool NORMED = false>
__device__ __forceinline__ void prep_issue(const bf16_t* src, const bf16_t* w, const float* cos_t, const float* sin_t,
                                           int pos, int half, int lane, PrepRegs<PER>& g) {
  __builtin_memcpy(g.x, src + lane * PER, sizeof g.x);
  if (NORMED || w) {
    __builtin_memcpy(g.w, w + lane * PER, sizeof g.w);
    const int hl = half / PER;
    const bool lowg = lane < hl, rot = lane < 2 * hl;
    // (a lane's entries lie side by side: one load each of the two tables; lanes that rotate nothing read the first ones)
    const size_t e = (size_t)pos * half + (rot ? (lowg ? lane : lane - hl) * PER : 0);
    __builtin_memcpy(g.c, cos_t + e, sizeof g.c);
    __builtin_memcpy(g.s, sin_t + e, sizeof g.s);
  }
}

template <int PER>
__device__ __forceinline__ void prep_finish(const PrepRegs<PER>& g, bool normed, int half, float eps, int lane,
                                            float (&x)[PER]) {
  constexpr int HD = 64 * PER;
#pragma unroll
  for (int i = 0; i < PER; ++i) x[i] = i & 1 ? dm_bf2f_hi(g.x[i >> 1]) : dm_bf2f_lo(g.x[i >> 1]);
  if (!normed) return;
  float a = 0.f;
#pragma unroll
  for (int i = 0; i < PER; ++i) a = dm_fma(x[i], x[i], a);
  const float inv = dm_rsqrt(dm_wave_sum<64>(a) / (float)HD + eps);
#pragma unroll
  for (int i = 0; i < PER; ++i) x[i] = dm_rb((i & 1 ? dm_bf2f_hi(g.w[i >> 1]) : dm_bf2f_lo(g.w[i >> 1])) * dm_rb(x[i] * inv));
  // rotate pairs (e, e + half), e < half; the partner channel lives hl lanes away
  const int hl = half / PER;
  const bool lowg = lane < hl, rot = lane < 2 * hl;
  const int partner = lowg ? lane + hl : lane - hl;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const float other = __shfl(x[i], partner & 63, 64);
    if (rot) {
      float r;
      if (lowg) {
        r = x[i] * g.c[i];
        r = dm_fma(-other, g.s[i], r);
      } else {
        r = other * g.s[i];
        r = dm_fma(x[i], g.c[i], r);
      }
      x[i] = r;  // rounded on store
    }
  }
}

// one wavefront per (head, token)
template <int PER>
__global__ __launch_bounds__(64) void attn_prep_kernel(PrepArgs p) {
  constexpr int HD = 64 * PER;
  const int hidx = blockIdx.x, t = blockIdx.y, lane = threadIdx.x;
  const int offset = p.d_offset ? *p.d_offset : p.offset;
  const int pos = offset + t;
  if (pos >= p.cap || pos >= p.npos) return;  // host checks the static case; device offset guarded here
  const bf16_t* src;
  bf16_t* dst;
  const bf16_t* w = nullptr;
  if (hidx < p.Hq) {
    src = p.qg + ((size_t)t * p.Hq + hidx) * 2 * HD;
    dst = p.q_rot + ((size_t)t * p.Hq + hidx) * HD;
    w = p.qw;
  } else if (hidx < p.Hq + p.Hkv) {
    const int h = hidx - p.Hq;
    src = p.kx + ((size_t)t * p.Hkv + h) * HD;
    dst = p.k_cache + ((size_t)h * p.cap + pos) * HD;
    w = p.kw;
  } else {
    const int h = hidx - p.Hq - p.Hkv;
    src = p.vx + ((size_t)t * p.Hkv + h) * HD;
    dst = p.v_cache + ((size_t)h * p.cap + pos) * HD;
  }
  PrepRegs<PER> g;
  prep_issue<PER>(src, w, p.cos_t, p.sin_t, pos, p.half, lane, g);
  float x[PER];
  prep_finish<PER>(g, w != nullptr, p.half, p.eps, lane, x);
#pragma unroll
  for (int i = 0; i < PER; ++i) dst[lane * PER + i] = dm_f2bf(x[i]);
}

struct SdpaArgs {
  const bf16_t* q_rot;   // [T, Hq, HD]
  const bf16_t* k_cache; // [Hkv, cap, HD]
  const bf16_t* v_cache;
  const bf16_t* qg;      // [T, Hq, 2*HD] (gate half read by the merge)
  const int* d_offset;
  float* part_m;         // [T, Hq, nblk]
  float* part_l;         // [T, Hq, nblk]
  float* part_o;         // [T, Hq, nblk, HD]
  bf16_t* out;           // [T, Hq*HD]
  int T, Hq, Hkv, offset, cap, nblk;
  float scale;
  int finish;  // 1: every row has a single key block, the partial kernel applies the merge's
               //    arithmetic itself and writes `out` (no merge launch follows)
  int by_die;  // the 1024-thread form's workgroups are numbered by die (sdpa_place)
};

// Which (key block, first of N heads, row) a workgroup of a linear grid works on.
// Workgroups go round the eight dies in order, and every die has an L2 of its own: with the block
// index running fastest the heads and rows that read one key / value block sit on different dies, each
// of which fetches it (nine rows at a 16 k context: 97 us against 82). So everything that reads one (block, KV head) is given to one die, next
// to each other in its order. false: past the end (the last round of dies is padded).
constexpr int kDies = 8, kManyHeads = 4;
template <int N>
__host__ __device__ __forceinline__ int sdpa_head_groups(const SdpaArgs& p) { return (p.Hq / p.Hkv + N - 1) / N; }
// the (block, KV head, first head, how many of the N exist, row) of this workgroup
template <int N>
__device__ __forceinline__ bool sdpa_place(const SdpaArgs& p, int& b, int& hk, int& hq0, int& nh, int& t) {
  const int group = p.Hq / p.Hkv, per = sdpa_head_groups<N>(p), sharers = per * p.T;
  const int die = blockIdx.x % kDies, n = blockIdx.x / kDies, round = n / sharers, s = n - round * sharers;
  const int pair = round * kDies + die;  // KV head fastest: the pairs of a short context on different dies
  if (pair >= p.nblk * p.Hkv) return false;
  b = pair / p.Hkv;
  hk = pair - b * p.Hkv;
  t = s / per;
  const int h = (s - t * per) * N;
  hq0 = hk * group + h;
  nh = min(N, group - h);
  return true;
}
template <int N>
unsigned sdpa_die_grid(const SdpaArgs& p) {
  return (unsigned)((p.nblk * p.Hkv + kDies - 1) / kDies * kDies * sdpa_head_groups<N>(p) * p.T);
}

// 1024 threads: one query head against one block of ATT_KB keys. Grid (nblk, Hq, T), with p.by_die sdpa_die_grid<1>.
//
// The sums: a key's score is one fma chain per 64 channels, the chains added pairwise
// ((c0 + c1) + (c2 + c3)); a channel's output over the block is one chain per 64 keys, added
// the same way. That gives every one of the 1024 threads a chain of 64 in both phases.
//
// The arithmetic is small and a trip to memory is long, so the whole block -- every key row
// and every value row -- is requested by the 16 wavefronts at once, in 16-byte pieces with
// eight lanes to a 128-byte line, before anything is computed. The rows then pass through
// LDS (keys as 64-channel panels with rows padded by 16 bytes to spread the banks; the values
// take the same memory over once the scores are done). Rows past the last valid key are not
// read, and the chains that would hold only such rows are not run.
constexpr int SDPA_NT = 1024;
constexpr int SDPA_KROW = 64 * 2 + 16;  // bytes of a staged 64-channel key row

// A native vector, not HIP's uint4 struct: arrays of the struct copied to LDS through casts are
// left in scratch memory by the compiler, arrays of this type stay in registers.
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

template <int HD>
constexpr int sdpa_stage_bytes() {
  constexpr int k = (HD / 64) * ATT_KB * SDPA_KROW, v = ATT_KB * HD * 2;
  return k > v ? k : v;
}

// (p0 + p1) + (p2 + p3) for N = 4, p0 + p1 for N = 2
template <int N>
__device__ __forceinline__ float sdpa_pair_tree(const float* p, int stride) {
  float t[N];
#pragma unroll
  for (int i = 0; i < N; ++i) t[i] = p[i * stride];
#pragma unroll
  for (int w = N; w > 1; w /= 2)
#pragma unroll
    for (int i = 0; i < w / 2; ++i) t[i] = t[2 * i] + t[2 * i + 1];
  return t[0];
}

//
// PREP: the launch also does attn_prep's work (the per-head norm, RoPE and the KV append), so
// that no prep launch precedes it: wavefront 0 makes the query row of this (row, head) from the
// raw projection, wavefronts 1 .. t + 1 the key rows of the call's new positions that lie in this
// block (they go into the staged block in place of the cache's rows, which are not yet written),
// the new value rows are read from the raw projection, and the workgroup of a KV group's first
// head stores its own row's key and value to the cache. Static offset, T <= 8.
template <int HD, bool PREP>
__global__ __launch_bounds__(SDPA_NT) __attribute__((amdgpu_waves_per_eu(4, 4))) void sdpa_partial_kernel(SdpaArgs p,
                                                                                                           PrepArgs q) {
  int b = blockIdx.x, hq = blockIdx.y, t = blockIdx.z, hk, one;
  if (p.by_die) {
    if (!sdpa_place<1>(p, b, hk, hq, one, t)) return;
  } else {
    hk = hq / (p.Hq / p.Hkv);
  }
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int offset = PREP ? p.offset : (p.d_offset ? *p.d_offset : p.offset);
  const int last = min(offset + t, p.cap - 1);
  if (b * ATT_KB > last) return;

  constexpr int PPR = HD / 8;                    // 16-byte pieces per row
  constexpr int RPU = SDPA_NT / PPR;             // value rows covered by one load per thread
  constexpr int NLD = ATT_KB / RPU;              // loads per thread for the block (keys: same count)
  constexpr int KC = 64, NKC = HD / KC, KROW = SDPA_KROW;
  constexpr int KPC = ATT_KB * (KC / 8) / SDPA_NT, KRS = SDPA_NT / (KC / 8);
  constexpr int VB = 64, NVB = ATT_KB / VB;
  static_assert(SDPA_NT % PPR == 0 && ATT_KB % RPU == 0 && KPC * NKC == NLD, "piece mapping");
  static_assert(ATT_KB == 256 && NKC <= 4 && NVB == 4 && HD <= 256, "chains of 64, four wavefronts a chain group");
  extern __shared__ __align__(16) unsigned char stage[];
  __shared__ __align__(16) float qs[HD];
  __shared__ float pr[ATT_KB];
  __shared__ float red[4];
  __shared__ float part[4 * 256];  // chain results: [panel][key], later [key group][channel]

  const int nvalid = min(ATT_KB, last - b * ATT_KB + 1);
  const int row0 = tid / PPR, piece = tid - row0 * PPR;    // values: rows row0 + RPU*u, piece column
  const int krow0 = tid / (KC / 8), kpc = tid % (KC / 8);  // keys: rows krow0 + KRS*i of every panel
  const bf16_t* kbase = p.k_cache + ((size_t)hk * p.cap + (size_t)b * ATT_KB) * HD;
  const bf16_t* vblk = p.v_cache + ((size_t)hk * p.cap + (size_t)b * ATT_KB) * HD + 8 * piece;
  u32x4 kreg[NLD], vreg[NLD];
  // PREP: this wavefront's row of the prep (0: none, 1: the query, 2: a new key row at kpos);
  // its few loads go out ahead of the block's, so that they are back first
  constexpr int PER = HD / 64;
  PrepRegs<PER> pg;
  int task = 0, kpos = 0;
  const bool first_of_group = hq % (p.Hq / p.Hkv) == 0;
  if constexpr (PREP) {
    if (wave == 0) {
      task = 1;
      prep_issue<PER>(q.qg + ((size_t)t * p.Hq + hq) * 2 * HD, q.qw, q.cos_t, q.sin_t, offset + t, q.half, lane, pg);
    } else if (wave <= t + 1 && (offset + wave - 1) / ATT_KB == b) {
      task = 2;
      kpos = offset + wave - 1;
      prep_issue<PER>(q.kx + ((size_t)(wave - 1) * p.Hkv + hk) * HD, q.kw, q.cos_t, q.sin_t, kpos, q.half, lane, pg);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // Rows past the last valid key are neither requested nor staged (a short context leaves most
  // of the block empty, and a request costs its slot in the compute unit's load path whether or
  // not the line is cached); what LDS holds in their place is never added to anything.
  // PREP: nor are the key rows of this call's positions, which come from their wavefronts.
  auto key_row_staged = [&](int r) { return r < nvalid && !(PREP && b * ATT_KB + r >= offset); };
#pragma unroll
  for (int c = 0; c < NKC; ++c)
#pragma unroll
    for (int i = 0; i < KPC; ++i) {
      const int r = krow0 + KRS * i;
      if (key_row_staged(r)) kreg[c * KPC + i] = *reinterpret_cast<const u32x4*>(kbase + (size_t)r * HD + c * KC + 8 * kpc);
    }
#pragma unroll
  for (int u = 0; u < NLD; ++u) {
    const int vr = row0 + RPU * u;
    if (vr >= nvalid) continue;
    const bf16_t* src = vblk + (size_t)vr * HD;
    // a position of this call: its value row is still in the projection's output
    if (PREP && b * ATT_KB + vr >= offset)
      src = q.vx + ((size_t)(b * ATT_KB + vr - offset) * p.Hkv + hk) * HD + 8 * piece;
    vreg[u] = *reinterpret_cast<const u32x4*>(src);
  }
  // the output gate of a finishing block is requested with everything else
  bf16_t gate_pre = 0;
  if (p.finish && tid < HD) gate_pre = p.qg[((size_t)t * p.Hq + hq) * 2 * HD + HD + tid];
  if constexpr (!PREP)
    if (tid < HD) qs[tid] = p.scale * dm_bf2f(p.q_rot[((size_t)t * p.Hq + hq) * HD + tid]);

  // scores: thread (key, panel) runs the chain over the panel's 64 channels
#pragma unroll
  for (int c = 0; c < NKC; ++c)
#pragma unroll
    for (int i = 0; i < KPC; ++i) {
      const int dest = krow0 + KRS * i;
      if (!key_row_staged(dest)) continue;
      *reinterpret_cast<u32x4*>(stage + c * (ATT_KB * KROW) + dest * KROW + 16 * kpc) = kreg[c * KPC + i];
    }
  if constexpr (PREP) {
    if (task) {
      float x[PER];
      prep_finish<PER>(pg, true, q.half, q.eps, lane, x);
      if (task == 1) {
#pragma unroll
        for (int i = 0; i < PER; ++i) qs[lane * PER + i] = p.scale * dm_bf2f(dm_f2bf(x[i]));  // q_rot is bf16
      } else {
        const int dest = kpos - b * ATT_KB, ch = lane * PER;
        bf16_t* row = reinterpret_cast<bf16_t*>(stage + (ch / KC) * (ATT_KB * KROW) + dest * KROW) + ch % KC;
        bf16_t* crow = q.k_cache + ((size_t)hk * p.cap + kpos) * HD + ch;
        const bool append = first_of_group && wave - 1 == t;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
          const bf16_t v = dm_f2bf(x[i]);
          row[i] = v;
          if (append) crow[i] = v;
        }
      }
    }
    // this row's value row to the cache (the thread that holds its piece unclamped)
    if (first_of_group && b == (offset + t) / ATT_KB) {
#pragma unroll
      for (int u = 0; u < NLD; ++u)
        if (b * ATT_KB + row0 + RPU * u == offset + t)
          *reinterpret_cast<u32x4*>(q.v_cache + ((size_t)hk * p.cap + offset + t) * HD + 8 * piece) = vreg[u];
    }
  }
  __syncthreads();
  // wavefront w takes panel w % 4 of keys [64 (w / 4), +64): a SIMD (wavefronts go round the four
  // in order) then holds one panel of every key group, and the groups past the last valid key
  // drop out of all four SIMDs alike
  const int grp = wave & 3, key = (wave >> 2) * 64 + lane;
  if (grp < NKC && (wave >> 2) * 64 < nvalid) {
    u32x4 kws[KC / 8];
#pragma unroll
    for (int i = 0; i < KC / 8; ++i)
      kws[i] = *reinterpret_cast<const u32x4*>(stage + grp * (ATT_KB * KROW) + key * KROW + 16 * i);
    // the panel's 64 query values: channel 16 g + l in lane l of every 16-lane row
    float qv[4], acc = 0.f;
#pragma unroll
    for (int g = 0; g < 4; ++g) qv[g] = qs[grp * KC + 16 * g + (lane & 15)];
#pragma unroll
    for (int i = 0; i < KC / 8; ++i) {
      const u32x4 kw = kws[i];
      const float kf[8] = {dm_bf2f_lo(kw.x), dm_bf2f_hi(kw.x), dm_bf2f_lo(kw.y), dm_bf2f_hi(kw.y),
                           dm_bf2f_lo(kw.z), dm_bf2f_hi(kw.z), dm_bf2f_lo(kw.w), dm_bf2f_hi(kw.w)};
      if (i & 1) dm_dot8<8>(acc, qv[i >> 1], kf);
      else dm_dot8<0>(acc, qv[i >> 1], kf);
    }
    part[grp * ATT_KB + key] = acc;
  }
  __syncthreads();
  // block max, probabilities, their sum (the first four wavefronts hold the keys)
  const bool valid = tid < nvalid;
  float sc = 0.f;
  if (tid < ATT_KB) {
    sc = sdpa_pair_tree<NKC>(part + tid, ATT_KB);
    const float m = dm_wave_max<64>(valid ? sc : -DM_INF);
    if (lane == 0) red[wave] = m;
  }
  __syncthreads();
  float mg = red[0];
  mg = red[1] > mg ? red[1] : mg;
  mg = red[2] > mg ? red[2] : mg;
  mg = red[3] > mg ? red[3] : mg;
  __syncthreads();
  if (tid < ATT_KB) {
    const float pv = valid ? dm_exp(sc - mg) : 0.f;
    pr[tid] = pv;
    const float ws = dm_wave_sum<64>(pv);
    if (lane == 0) red[wave] = ws;
  }
  // values: thread (channel, group of 64 keys) runs the chain over the group's valid keys
  bf16_t (*vst)[HD] = reinterpret_cast<bf16_t (*)[HD]>(stage);
  // (up to the end of the last chain that runs, zeros past the last key: its probabilities are 0)
  const int nstage = (nvalid + VB - 1) / VB * VB;
#pragma unroll
  for (int u = 0; u < NLD; ++u) {
    const int r = row0 + RPU * u;
    if (r < nstage) *reinterpret_cast<u32x4*>(&vst[r][8 * piece]) = r < nvalid ? vreg[u] : u32x4{0, 0, 0, 0};
  }
  __syncthreads();  // probabilities and value rows in place (the key panels were last read two barriers ago)
  // two channels a thread
  const int ch = 2 * (tid % (HD / 2)), vg = tid / (HD / 2);
  if (vg < NVB && VB * vg >= nvalid) part[vg * HD + ch] = part[vg * HD + ch + 1] = 0.f;  // a chain with no valid key
  if (vg < NVB && VB * vg < nvalid) {
    float o[2] = {0.f, 0.f};
    auto sixteen = [&](auto gc) {
      constexpr int G = decltype(gc)::value;
      const float w = pr[VB * vg + 16 * G + (lane & 15)];
      uint32_t raw[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) raw[u] = *reinterpret_cast<const uint32_t*>(&vst[VB * vg + 16 * G + u][ch]);
      auto four = [&](auto bc) {
        constexpr int B = decltype(bc)::value;
        float v[4][2];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          v[u][0] = dm_bf2f_lo(raw[B + u]);
          v[u][1] = dm_bf2f_hi(raw[B + u]);
        }
        dm_axpy4<B>(o, w, v);
      };
      four(std::integral_constant<int, 0>{});
      four(std::integral_constant<int, 4>{});
      four(std::integral_constant<int, 8>{});
      four(std::integral_constant<int, 12>{});
    };
    sixteen(std::integral_constant<int, 0>{});
    sixteen(std::integral_constant<int, 1>{});
    sixteen(std::integral_constant<int, 2>{});
    sixteen(std::integral_constant<int, 3>{});
    part[vg * HD + ch] = o[0];
    part[vg * HD + ch + 1] = o[1];
  }
  __syncthreads();
  const size_t pi = ((size_t)t * p.Hq + hq) * p.nblk + b;
  float l = red[0] + red[1];
  l = l + red[2];
  l = l + red[3];
  if (p.finish) {
    // the merge over one block, operation for operation (sdpa_merge_kernel with nb == 1)
    if (tid < HD) {
      const float w = dm_exp(mg - mg);
      const float L = dm_fma(l, w, 0.f);
      const float O = dm_fma(sdpa_pair_tree<NVB>(part + tid, HD), w, 0.f);
      const float att = dm_rb(O / L);
      const float g = dm_sigmoid_bf16(dm_bf2f(gate_pre));
      p.out[((size_t)t * p.Hq + hq) * HD + tid] = dm_f2bf(g * att);
    }
    return;
  }
  if (tid < HD) p.part_o[pi * HD + tid] = sdpa_pair_tree<NVB>(part + tid, HD);
  if (tid == 0) {
    p.part_m[pi] = mg;
    p.part_l[pi] = l;
  }
}

// The same partial sums when there are many blocks to work through (long contexts): several
// workgroups resident per compute unit, and four query heads of a KV group in each, so that the key
// and value block is read once for the four.
//
// The arithmetic, fp32 chains of 64 whose order is fixed, is what bounds a block, and it runs on the
// matrix cores all the same: v_mfma_f32_4x4x1_16b_f32 adds one product to every element with one
// rounding (K = 1: the fused multiply-add of the chain's next step, bit for bit), 64 keys or channels
// by four heads an instruction. The heads' side (queries, later probabilities) is broadcast inside the
// instruction (cbsz = 4: every block takes the four values of block abid), so a register holds 16 steps
// of it. Eight clocks for 256 multiply-adds where vector instructions take 11 to 20 (two to four
// wavefronts a SIMD; a wavefront alone on its SIMD issues one every eight clocks).
//
// Scores: lane = key; wavefronts 0 - 3 run the lower half of the 64-channel chains, 4 - 7 the upper
// half, the key block reaching them through LDS a chain of each at a time (global loads of whole
// 128-byte pieces). Values: a wavefront has one 64-key chain of half the channels, two a lane; the
// four chains of a channel meet in LDS. Every sum of every head keeps its order.
// us before (256 threads, vector fmas, queries read from LDS) -> now, two KV groups of eight heads of 256:
// 4 rows at 6621 keys 23.7 -> 17.4, 2 at 9000 23.2 -> 17.0, 6 at 1445 19.3 -> 12.3, 9 at 16000 117 -> 62.
// (A KV group that is no multiple of four heads repeats its last one; what that makes is not stored. What
// it costs stands at the choice of the form, sdpa_decode.)
// grid sdpa_die_grid<kManyHeads>, 512 threads
template <int HD>
__global__ __launch_bounds__(512, 4) void sdpa_partial_many_kernel(SdpaArgs p) {
  constexpr int NH = kManyHeads, NT = 512;
  int b, hk, hq0, nh, t;
  if (!sdpa_place<kManyHeads>(p, b, hk, hq0, nh, t)) return;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int offset = p.d_offset ? *p.d_offset : p.offset;
  const int last = min(offset + t, p.cap - 1);
  if (b * ATT_KB > last) return;
  constexpr int NKC = HD / 64, NVB = ATT_KB / 64, KLD = 64 + 8, STEPS = NKC / 2;
  static_assert(ATT_KB == 256, "four wavefronts of keys");
  static_assert(NKC == 2 || NKC == 4, "head widths of 128 and 256");
  typedef float f32x4 __attribute__((ext_vector_type(4)));

  // the key panels; before them the queries, after them the halves' score sums and the value chains
  __shared__ __align__(16) bf16_t ks[2][ATT_KB][KLD];
  __shared__ float pr[NH][ATT_KB];
  __shared__ float red[NH][4];
  float* const part = reinterpret_cast<float*>(ks);  // [NH][NVB * HD]
  static_assert(sizeof(ks) >= NH * NVB * HD * 4, "the value chains fit where the keys were");

  const int half = wave >> 2, row = (wave & 3) * 64 + lane;  // of the scores: chains of this half, this key
  const int j0 = 2 * half;                                   // of the softmax: heads j0, j0 + 1
  const bool valid = b * ATT_KB + row <= last;
  const int nvalid = min(ATT_KB, last - b * ATT_KB + 1);
  // (rows past the last key read as zeros: their scores are masked, their probabilities 0)
  const size_t blk0 = ((size_t)hk * p.cap + (size_t)b * ATT_KB) * HD;
  const __amdgpu_buffer_rsrc_t kbuf = dm_buffer(p.k_cache + blk0, nvalid * HD * 2), vbuf = dm_buffer(p.v_cache + blk0, nvalid * HD * 2);

  // step s: panels s and s + STEPS, 4096 16-byte pieces. All of a step travels in registers ahead of
  // its use, and so do the first 32 keys of this thread's value chain: a block is a chain of memory
  // latencies otherwise.
  u32x4 kreg[8];
  auto fetch_keys = [&](int s) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int idx = tid + NT * (u & 3);
      kreg[u] = __builtin_amdgcn_raw_buffer_load_b128(kbuf, (idx >> 3) * (HD * 2) + 16 * (idx & 7) + 128 * (s + STEPS * (u >> 2)), 0, 0);
    }
  };
  fetch_keys(0);
  constexpr int TPC = HD / 2;  // threads a value chain
  const int vg = tid / TPC, vcg = tid % TPC;
  const bool holds = vg < NVB;  // (whole wavefronts)
  uint32_t vreg[2][16];
  auto fetch_values = [&](auto set, int i0) {
    constexpr int S = decltype(set)::value;
    if (holds) {
#pragma unroll
      for (int u = 0; u < 16; ++u)
        vreg[S][u] = __builtin_amdgcn_raw_buffer_load_b32(vbuf, (64 * vg + i0 + u) * (HD * 2) + 4 * vcg, 0, 0);
    }
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  fetch_values(S0{}, 0);
  fetch_values(S1{}, 16);
  // this half's query channels: 16 g + a of head i in lane 4 a + i
  constexpr int QG = HD / 32;
  float q[QG];
  {
    const bf16_t* qrow = p.q_rot + ((size_t)t * p.Hq + hq0 + min(lane & 3, nh - 1)) * HD + half * (HD / 2) + (lane >> 2);
#pragma unroll
    for (int g = 0; g < QG; ++g) q[g] = p.scale * dm_bf2f(qrow[16 * g]);
  }
  auto step16 = [&](f32x4 acc, float qv, const float (&k)[16]) {
#define ORN_STEP(A) acc = __builtin_amdgcn_mfma_f32_4x4x1f32(qv, k[A], acc, 4, A, 0);
    ORN_STEP(0) ORN_STEP(1) ORN_STEP(2) ORN_STEP(3) ORN_STEP(4) ORN_STEP(5) ORN_STEP(6) ORN_STEP(7)
    ORN_STEP(8) ORN_STEP(9) ORN_STEP(10) ORN_STEP(11) ORN_STEP(12) ORN_STEP(13) ORN_STEP(14) ORN_STEP(15)
#undef ORN_STEP
    return acc;
  };
  f32x4 chain[STEPS];
  auto scores = [&](auto sc) {
    constexpr int s = decltype(sc)::value;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int idx = tid + NT * (u & 3);
      *reinterpret_cast<u32x4*>(&ks[u >> 2][idx >> 3][8 * (idx & 7)]) = kreg[u];
    }
    __syncthreads();
    if constexpr (s + 1 < STEPS) fetch_keys(s + 1);
    chain[s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float k[16];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const uint4 kw = *reinterpret_cast<const uint4*>(&ks[half][row][16 * g + 8 * h]);
        const uint32_t w[4] = {kw.x, kw.y, kw.z, kw.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          k[8 * h + 2 * e] = dm_bf2f_lo(w[e]);
          k[8 * h + 2 * e + 1] = dm_bf2f_hi(w[e]);
        }
      }
      chain[s] = step16(chain[s], q[4 * s + g], k);
    }
    __syncthreads();
  };
  scores(S0{});
  if constexpr (STEPS == 2) scores(S1{});
  // (c0 + c1) + (c2 + c3): each half hands the other the two heads it does not go on with
  f32x4 sum = chain[0];
  if constexpr (STEPS == 2) sum = chain[0] + chain[1];
  float* const other = part + row;
#pragma unroll
  for (int j = 0; j < 2; ++j) other[((half ^ 1) * 2 + j) * ATT_KB] = half ? sum[j] : sum[2 + j];
  __syncthreads();
  float sc[2], mg[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const float mine = half ? sum[2 + j] : sum[j], theirs = other[(j0 + j) * ATT_KB];
    sc[j] = mine + theirs;
    const float m = dm_wave_max<64>(valid ? sc[j] : -DM_INF);  // block max
    if (lane == 0) red[j0 + j][wave & 3] = m;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const float* r = red[j0 + j];
    float m = r[0];
    m = r[1] > m ? r[1] : m;
    m = r[2] > m ? r[2] : m;
    m = r[3] > m ? r[3] : m;
    mg[j] = m;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const float pv = valid ? dm_exp(sc[j] - mg[j]) : 0.f;
    pr[j0 + j][row] = pv;
    const float ws = dm_wave_sum<64>(pv);
    if (lane == 0) red[j0 + j][wave & 3] = ws;
    if (row == 0 && j0 + j < nh) p.part_m[((size_t)t * p.Hq + hq0 + j0 + j) * p.nblk + b] = mg[j];
  }
  __syncthreads();
  // values: chain vg = keys 64 * vg .. + 64, channels 2 vcg, 2 vcg + 1 of the four heads
  if (holds) {
    f32x4 o0 = {0.f, 0.f, 0.f, 0.f}, o1 = o0;
    auto batch = [&](auto set, int g) {
      constexpr int S = decltype(set)::value;
      const float w = pr[lane & 3][64 * vg + 16 * g + (lane >> 2)];  // key a of head i in lane 4 a + i
#define ORN_KEY(A)                                                                                  \
  o0 = __builtin_amdgcn_mfma_f32_4x4x1f32(w, dm_bf2f_lo(vreg[S][A]), o0, 4, A, 0);                  \
  o1 = __builtin_amdgcn_mfma_f32_4x4x1f32(w, dm_bf2f_hi(vreg[S][A]), o1, 4, A, 0);
      ORN_KEY(0) ORN_KEY(1) ORN_KEY(2) ORN_KEY(3) ORN_KEY(4) ORN_KEY(5) ORN_KEY(6) ORN_KEY(7)
      ORN_KEY(8) ORN_KEY(9) ORN_KEY(10) ORN_KEY(11) ORN_KEY(12) ORN_KEY(13) ORN_KEY(14) ORN_KEY(15)
#undef ORN_KEY
    };
    batch(S0{}, 0);
    fetch_values(S0{}, 32);
    batch(S1{}, 1);
    fetch_values(S1{}, 48);
    batch(S0{}, 2);
    batch(S1{}, 3);
#pragma unroll
    for (int j = 0; j < NH; ++j)
      *reinterpret_cast<float2*>(&part[j * (NVB * HD) + vg * HD + 2 * vcg]) = make_float2(o0[j], o1[j]);
  }
  __syncthreads();
  for (int i = tid; i < nh * HD; i += NT) {
    const int j = i / HD, d = i - j * HD;
    p.part_o[(((size_t)t * p.Hq + hq0 + j) * p.nblk + b) * HD + d] = sdpa_pair_tree<NVB>(part + j * (NVB * HD) + d, HD);
  }
  if (tid < nh) {
    float l = red[tid][0] + red[tid][1];
    l = l + red[tid][2];
    l = l + red[tid][3];
    p.part_l[((size_t)t * p.Hq + hq0 + tid) * p.nblk + b] = l;
  }
}

// The same again for eight query heads of a KV group a workgroup and one workgroup a compute unit: half as many workgroups as the
// four-head form has, for calls where those are more than the compute units and share them.
//
// What bounds a block here is issue. A load instruction takes the compute unit's address path 16 clocks whatever its width:
// the block as 16 bytes a lane straight into LDS (keys) and 8 a lane into registers (values, four channels) is 384 of them,
// 2.7 us. (The keys' requests are in the buffer form: behind one in the global form the compiler waits for every load in
// flight where it means to wait for one.) The arithmetic is that of the four-head form, two quads of heads as independent
// chains: 4096 instructions of eight clocks on four matrix cores, 4 us. The bf16 operands are unpacked 16 steps ahead,
// between the products (right ahead of its own, each waits out the hazard between the two).
//
// Scores: lane = key; wavefronts 0 - 3 run the lower half of the 64-channel chains, 4 - 7 the upper half; a key's eight
// pieces of a panel lie permuted in LDS (piece i at i ^ (key & 7)), so that eight keys' reads are on different banks.
// Values: wavefront w of the first four has the 64-key chain w of all channels; the four chains of a channel
// meet in LDS. Every sum of every head keeps its order. (A KV group that is no multiple of eight heads repeats its last one; what
// that makes is not stored.)
//
// PREP: attn_prep's work too: wavefront w makes query head w and the key row of the call's w-th new position in the block, new value
// rows are read from the raw projection, and of the workgroups of a row's last block each stores its query heads, the one of a KV
// group's first heads also the row's key and value. Static offset, T <= 8.
// grid sdpa_die_grid<kEightHeads>, 512 threads
constexpr int kEightHeads = 8;
template <int HD>
constexpr int sdpa_eight_bytes() { return (HD / 64) * ATT_KB * 128; }
template <int HD, bool PREP>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void sdpa_partial_eight_kernel(SdpaArgs p, PrepArgs pq) {
  constexpr int NH = kEightHeads, NQ = NH / 4, HPW = NH / 2;  // heads of the workgroup; of a half in the softmax
  int b, hk, hq0, nh, t;
  if (!sdpa_place<NH>(p, b, hk, hq0, nh, t)) return;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int offset = PREP ? p.offset : (p.d_offset ? *p.d_offset : p.offset);
  const int last = min(offset + t, p.cap - 1);
  if (b * ATT_KB > last) return;
  constexpr int NKC = HD / 64, NVB = ATT_KB / 64, STEPS = NKC / 2, PER = HD / 64, PANEL = ATT_KB * 128;
  static_assert(ATT_KB == 256, "four wavefronts of keys");
  static_assert(NKC == 2 || NKC == 4, "head widths of 128 and 256");
  typedef float f32x4 __attribute__((ext_vector_type(4)));

  // the key panels; after them the halves' score sums and the value chains
  extern __shared__ __align__(16) unsigned char stage[];
  __shared__ float pr[NH][ATT_KB];                       // probabilities; before them the queries
  __shared__ float red[NH][4], redm[NH][4];              // the key groups' sums and maxima
  float* const part = reinterpret_cast<float*>(stage);   // [NH][NVB * HD]
  static_assert(sdpa_eight_bytes<HD>() >= NH * NVB * HD * 4, "the value chains fit where the keys were");
  float* const qsh = &pr[0][0];                          // PREP: [NH][HD]
  static_assert(HD <= ATT_KB, "the queries fit where the probabilities will be");

  const int half = wave >> 2, row = (wave & 3) * 64 + lane;  // of the scores: chains of this half, this key
  const int j0 = HPW * half;                                 // of the softmax: heads j0 ..
  const bool valid = b * ATT_KB + row <= last;
  const int nvalid = min(ATT_KB, last - b * ATT_KB + 1);
  // rows that the cache has; the others are this call's
  const int nold = PREP ? min(nvalid, max(0, offset - b * ATT_KB)) : nvalid;
  const size_t blk0 = ((size_t)hk * p.cap + (size_t)b * ATT_KB) * HD;
  const __amdgpu_buffer_rsrc_t vbuf = dm_buffer(p.v_cache + blk0, nold * HD * 2);

  // PREP: the few loads of this wavefront's rows go out ahead of the block's
  PrepRegs<PER> pgq, pgk;
  const int kpos = max(offset, b * ATT_KB) + wave;  // the call's position this wavefront makes the key row of
  const bool has_k = PREP && kpos < b * ATT_KB + nvalid;
  if constexpr (PREP) {
    prep_issue<PER, true>(pq.qg + ((size_t)t * p.Hq + hq0 + min(wave, nh - 1)) * 2 * HD, pq.qw, pq.cos_t, pq.sin_t, offset + t, pq.half, lane, pgq);
    const int kp = min(kpos, offset + p.T - 1);
    prep_issue<PER, true>(pq.kx + ((size_t)(kp - offset) * p.Hkv + hk) * HD, pq.kw, pq.cos_t, pq.sin_t, kp, pq.half, lane, pgk);
    __builtin_amdgcn_sched_barrier(0);
  }
  // this half's query channels: 16 g + a of head i of a quad in lane 4 a + i
  constexpr int QG = HD / 32;
  float q[NQ][QG];
  bf16_t qraw[NQ][QG];
  if constexpr (!PREP) {
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
      const bf16_t* qrow = p.q_rot + ((size_t)t * p.Hq + hq0 + min(4 * n + (lane & 3), nh - 1)) * HD + half * (HD / 2) + (lane >> 2);
#pragma unroll
      for (int g = 0; g < QG; ++g) qraw[n][g] = qrow[16 * g];
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // keys: 8 rows of a panel, 1 KB, a load; rows that the cache does not have repeat another (they are masked, or written
  // below). (No load stands under a condition that others could be counted past.)
  {
    const __amdgpu_buffer_rsrc_t kbuf = dm_buffer(p.k_cache + blk0, max(nold, 1) * HD * 2);
#pragma unroll
    for (int i = 0; i < NKC * 4; ++i) {
      const int c = wave + 8 * (i & 3), panel = i >> 2, r = min(8 * c + (lane >> 3), max(nold, 1) - 1);
      typedef __attribute__((address_space(3))) void lds_t;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(kbuf, (lds_t*)(stage + panel * PANEL + c * 1024), 16,
                                               r * (HD * 2) + panel * 128 + 16 * ((lane & 7) ^ (lane >> 3)), 0, 0, 0);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  // values: PER channels a lane, the first half of the chain's keys right behind the block's keys
  typedef uint32_t vrow_t __attribute__((ext_vector_type(PER / 2)));
  const bool holds = wave < NVB;
  vrow_t vreg[4][16];
  auto load_row = [&](const __amdgpu_buffer_rsrc_t& buf, int at) {
    vrow_t v;
    if constexpr (PER == 4) {
      v = __builtin_bit_cast(vrow_t, __builtin_amdgcn_raw_buffer_load_b64(buf, at + 8 * lane, 0, 0));
    } else {
      v[0] = __builtin_amdgcn_raw_buffer_load_b32(buf, at + 4 * lane, 0, 0);
    }
    return v;
  };
  auto fetch_values = [&](auto set) {
    constexpr int S = decltype(set)::value;
#pragma unroll
    for (int u = 0; u < 16; ++u) vreg[S][u] = load_row(vbuf, (64 * wave + 16 * S + u) * (HD * 2));
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  using S2 = std::integral_constant<int, 2>;
  using S3 = std::integral_constant<int, 3>;
  uint32_t qrow[PER / 2], krow[PER / 2];
  auto heads = [&](auto path) {  // (the paths' tags keep the compiler from doing it ahead of the requests, where the paths agree)
    if constexpr (PREP) {
      float x[PER];
#pragma unroll
      for (int i = 0; i < PER / 2; ++i) asm volatile("; rows on path %4" : "+v"(pgq.x[i]), "+v"(pgk.x[i]), "+v"(pgq.w[i]), "+v"(pgk.w[i]) : "n"(decltype(path)::value));
      prep_finish<PER>(pgq, true, pq.half, pq.eps, lane, x);
#pragma unroll
      for (int e = 0; e < PER; e += 2) {  // q_rot is bf16
        qrow[e / 2] = dm_f2bf2(x[e], x[e + 1]);
        qsh[wave * HD + lane * PER + e] = p.scale * dm_bf2f_lo(qrow[e / 2]);
        qsh[wave * HD + lane * PER + e + 1] = p.scale * dm_bf2f_hi(qrow[e / 2]);
      }
      if (has_k) {
        prep_finish<PER>(pgk, true, pq.half, pq.eps, lane, x);
#pragma unroll
        for (int e = 0; e < PER; e += 2) krow[e / 2] = dm_f2bf2(x[e], x[e + 1]);
      }
    } else {
#pragma unroll
      for (int n = 0; n < NQ; ++n)
#pragma unroll
        for (int g = 0; g < QG; ++g) q[n][g] = p.scale * dm_bf2f(qraw[n][g]);
    }
  };
  if (holds) {
    fetch_values(S0{});
    fetch_values(S1{});
    __builtin_amdgcn_sched_barrier(0);
    heads(S1{});
  } else {
    heads(S0{});
  }
  // this wavefront's part of the keys is here (the values behind it are not)
  asm volatile("" ::: "memory");
  if (holds) __builtin_amdgcn_s_waitcnt(0x0070 | (32 >> 4) << 14);  // at most 32 loads left, every LDS access done
  else __builtin_amdgcn_s_waitcnt(0x0070);
  __builtin_amdgcn_s_barrier();  // (__syncthreads would wait for the values too)
  asm volatile("" ::: "memory");
  if constexpr (PREP) {
    if (nold < nvalid) {  // (of the whole workgroup)
      if (has_k) {
        const int r = kpos - b * ATT_KB, ch = lane * PER, at = ch % 64 * 2;
#pragma unroll
        for (int e = 0; e < PER / 2; ++e)
          *reinterpret_cast<uint32_t*>(stage + ch / 64 * PANEL + r * 128 + ((at & ~15) ^ ((r & 7) << 4)) + (at & 15) + 4 * e) = krow[e];
      }
      __syncthreads();
    }
#pragma unroll
    for (int n = 0; n < NQ; ++n)
#pragma unroll
      for (int g = 0; g < QG; ++g) q[n][g] = qsh[(4 * n + (lane & 3)) * HD + half * (HD / 2) + 16 * g + (lane >> 2)];
  }
  if (holds) {
    fetch_values(S2{});
    fetch_values(S3{});
  }
  __builtin_amdgcn_sched_barrier(0);
  f32x4 sum[NQ];
#pragma unroll
  for (int s = 0; s < STEPS; ++s) {
    f32x4 chain[NQ];
#pragma unroll
    for (int n = 0; n < NQ; ++n) chain[n] = f32x4{0.f, 0.f, 0.f, 0.f};
    uint4 kw[8];
    const unsigned char* const kr = stage + (half * STEPS + s) * PANEL + row * 128;
#pragma unroll
    for (int i = 0; i < 8; ++i) kw[i] = *reinterpret_cast<const uint4*>(kr + 16 * (i ^ (lane & 7)));
    auto channel = [&](int i) {
      const uint4& w = kw[i >> 3];
      const uint32_t u[4] = {w.x, w.y, w.z, w.w};
      return i & 1 ? dm_bf2f_hi(u[(i >> 1) & 3]) : dm_bf2f_lo(u[(i >> 1) & 3]);
    };
    float k[2][16];
#pragma unroll
    for (int i = 0; i < 16; ++i) k[0][i] = channel(i);
    __builtin_amdgcn_sched_barrier(0);
    auto sixteen = [&](auto gc) {
      constexpr int G = decltype(gc)::value;
#define ORN_STEP(A)                                                                                                  \
  _Pragma("unroll") for (int n = 0; n < NQ; ++n)                                                                     \
      chain[n] = __builtin_amdgcn_mfma_f32_4x4x1f32(q[n][4 * s + G], k[G & 1][A], chain[n], 4, A, 0);                \
  if constexpr (G < 3) k[(G & 1) ^ 1][A] = channel((16 * G + 16 + A) & 63);
      ORN_STEP(0) ORN_STEP(1) ORN_STEP(2) ORN_STEP(3) ORN_STEP(4) ORN_STEP(5) ORN_STEP(6) ORN_STEP(7)
      ORN_STEP(8) ORN_STEP(9) ORN_STEP(10) ORN_STEP(11) ORN_STEP(12) ORN_STEP(13) ORN_STEP(14) ORN_STEP(15)
#undef ORN_STEP
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, NQ, 0);
        if constexpr (G < 3) __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    sixteen(S0{});
    sixteen(S1{});
    sixteen(S2{});
    sixteen(S3{});
#pragma unroll
    for (int n = 0; n < NQ; ++n) sum[n] = s == 0 ? chain[n] : sum[n] + chain[n];
  }
  // PREP: the values of the call's own positions up to this row's come from the projection; this row goes to the cache, its
  // query heads to q_rot
  if constexpr (PREP) {
    if (holds && nold < nvalid) {
      const __amdgpu_buffer_rsrc_t xbuf = dm_buffer(pq.vx + (size_t)hk * HD, (uint32_t)(t * p.Hkv + 1) * (HD * 2));
      const int x0 = max(offset, b * ATT_KB) - offset - nold;
#pragma unroll
      for (int u = 0; u < 64; ++u) {
        const int r = 64 * wave + u;
        if (r >= nold && r < nvalid) vreg[u >> 4][u & 15] = load_row(xbuf, (x0 + r) * (p.Hkv * HD * 2));
      }
    }
    if (b == last / ATT_KB && wave < nh)
      __builtin_memcpy(pq.q_rot + ((size_t)t * p.Hq + hq0 + wave) * HD + lane * PER, qrow, sizeof qrow);  // (as the caller has aligned it)
    if (hq0 == hk * (p.Hq / p.Hkv) && has_k && kpos == last) {
#pragma unroll
      for (int e = 0; e < PER / 2; ++e) {
        const size_t at = ((size_t)hk * p.cap + last) * HD + lane * PER + 2 * e;
        *reinterpret_cast<uint32_t*>(pq.k_cache + at) = krow[e];
        *reinterpret_cast<uint32_t*>(pq.v_cache + at) =
            *reinterpret_cast<const uint32_t*>(pq.vx + ((size_t)t * p.Hkv + hk) * HD + lane * PER + 2 * e);
      }
    }
  }
  __syncthreads();  // the keys have been read
  // (c0 + c1) + (c2 + c3): each half hands the other the heads it does not go on with
  auto head_sum = [&](int j) { return sum[j >> 2][j & 3]; };
  float* const other = part + row;
#pragma unroll
  for (int j = 0; j < HPW; ++j) other[((half ^ 1) * HPW + j) * ATT_KB] = half ? head_sum(j) : head_sum(HPW + j);
  __syncthreads();
  float sc[HPW], mg[HPW];
#pragma unroll
  for (int j = 0; j < HPW; ++j) {
    const float mine = half ? head_sum(HPW + j) : head_sum(j), theirs = other[(j0 + j) * ATT_KB];
    sc[j] = mine + theirs;
    const float m = dm_wave_max<64>(valid ? sc[j] : -DM_INF);  // block max
    if (lane == 0) redm[j0 + j][wave & 3] = m;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < HPW; ++j) {
    const float* r = redm[j0 + j];
    float m = r[0];
    m = r[1] > m ? r[1] : m;
    m = r[2] > m ? r[2] : m;
    m = r[3] > m ? r[3] : m;
    mg[j] = m;
    const float pv = valid ? dm_exp(sc[j] - m) : 0.f;
    pr[j0 + j][row] = pv;
    const float ws = dm_wave_sum<64>(pv);
    if (lane == 0) red[j0 + j][wave & 3] = ws;
    if (row == 0 && j0 + j < nh) p.part_m[((size_t)t * p.Hq + hq0 + j0 + j) * p.nblk + b] = m;
  }
  __syncthreads();
  // values: chain `wave` = keys 64 * wave .. + 64, PER channels of the heads
  if (holds) {
    f32x4 o[PER][NQ];
#pragma unroll
    for (int c = 0; c < PER; ++c)
#pragma unroll
      for (int n = 0; n < NQ; ++n) o[c][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    float w[NQ][4];  // key a of head i of sixteen in lane 4 a + i
#pragma unroll
    for (int n = 0; n < NQ; ++n)
#pragma unroll
      for (int g = 0; g < 4; ++g) w[n][g] = pr[4 * n + (lane & 3)][64 * wave + 16 * g + (lane >> 2)];
    constexpr int AHEAD = 4;  // keys unpacked ahead
    float v[2][AHEAD][PER];
    auto unpack = [&](int e, int i) {  // key i of the e-th four
      const vrow_t u = vreg[e >> 2][4 * (e & 3) + i];
#pragma unroll
      for (int c = 0; c < PER; ++c) v[e & 1][i][c] = c & 1 ? dm_bf2f_hi(u[c >> 1]) : dm_bf2f_lo(u[c >> 1]);
    };
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) unpack(0, i);
    __builtin_amdgcn_sched_barrier(0);
    auto four = [&](auto ec) {
      constexpr int E = decltype(ec)::value;
#define ORN_KEY(A)                                                                                                         \
  _Pragma("unroll") for (int c = 0; c < PER; ++c) _Pragma("unroll") for (int n = 0; n < NQ; ++n)                            \
      o[c][n] = __builtin_amdgcn_mfma_f32_4x4x1f32(w[n][E >> 2], v[E & 1][A][c], o[c][n], 4, 4 * (E & 3) + A, 0);           \
  if constexpr (E < 15) unpack((E + 1) & 15, A);
      ORN_KEY(0) ORN_KEY(1) ORN_KEY(2) ORN_KEY(3)
#undef ORN_KEY
#pragma unroll
      for (int i = 0; i < 4 * PER; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, NQ, 0);
        if constexpr (E < 15) __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
#define ORN_FOURS(E) four(std::integral_constant<int, E>{}); four(std::integral_constant<int, E + 1>{}); \
                     four(std::integral_constant<int, E + 2>{}); four(std::integral_constant<int, E + 3>{});
    ORN_FOURS(0) ORN_FOURS(4) ORN_FOURS(8) ORN_FOURS(12)
#undef ORN_FOURS
#pragma unroll
    for (int n = 0; n < NQ; ++n)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float* const to = &part[(4 * n + j) * (NVB * HD) + wave * HD + PER * lane];
        if constexpr (PER == 4)
          *reinterpret_cast<float4*>(to) = make_float4(o[0][n][j], o[1][n][j], o[PER - 2][n][j], o[PER - 1][n][j]);
        else
          *reinterpret_cast<float2*>(to) = make_float2(o[0][n][j], o[1][n][j]);
      }
  }
  __syncthreads();
  for (int i = tid; i < nh * HD; i += 512) {
    const int j = i / HD, d = i - j * HD;
    p.part_o[(((size_t)t * p.Hq + hq0 + j) * p.nblk + b) * HD + d] = sdpa_pair_tree<NVB>(part + j * (NVB * HD) + d, HD);
  }
  if (tid < nh) {
    float l = red[tid][0] + red[tid][1];
    l = l + red[tid][2];
    l = l + red[tid][3];
    p.part_l[((size_t)t * p.Hq + hq0 + tid) * p.nblk + b] = l;
  }
}

// Merge: blocks ascending, divide, gate. Grid (Hq, T), one wavefront a row, HD / 64 channels a lane.
// A few trips to memory and little else: lane b fetches block b's maximum and sum, every lane asks for its
// channels' partial outputs of up to kMergeAhead blocks in the same trip, and the block weights exp(m_b - M) are made once (lane b)
// and read from its lane; the sums over the blocks stay one ascending fma chain a channel. A load
// takes the address path 16 clocks whatever its width, so a lane takes all its channels in one. As HD / 64 wavefronts of
// one channel a lane, which asked for the outputs behind the maxima and for 32 blocks whatever the row had, us a launch, before / now: one
// row, 10 blocks 4.0 / 2.9, 63 blocks 5.6 / 4.8, two rows of 24 blocks 4.0 / 3.6, four rows of 27 4.0 / 3.9; whole calls, one row, 2 blocks
// 12.2 / 10.8, 6 blocks 12.9 / 11.1, 36 blocks 19.0 / 17.3.
constexpr int kMergeAhead = 32;
template <int HD>
__global__ __launch_bounds__(64) void sdpa_merge_kernel(SdpaArgs p) {
  constexpr int PER = HD / 64, SET = 8;
  typedef float chan_t __attribute__((ext_vector_type(PER)));
  typedef uint32_t bits_t __attribute__((ext_vector_type(PER / 2)));
  const int h = blockIdx.x, t = blockIdx.y, lane = threadIdx.x;
  const int offset = p.d_offset ? *p.d_offset : p.offset;
  const int last = min(offset + t, p.cap - 1);
  const int nb = last / ATT_KB + 1;
  const size_t pi = ((size_t)t * p.Hq + h) * p.nblk;
  const float *pm = p.part_m + pi, *pl = p.part_l + pi, *po = p.part_o + pi * HD + PER * lane;
  float mb = pm[min(lane, nb - 1)], lb = pl[min(lane, nb - 1)];
  chan_t v[kMergeAhead];
  auto fetch = [&](int b0) {  // sets of blocks that the row has (the last one repeats its last block)
#pragma unroll
    for (int s = 0; s < kMergeAhead; s += SET)
      if (b0 + s < nb)
#pragma unroll
        for (int u = s; u < s + SET; ++u) v[u] = *reinterpret_cast<const chan_t*>(po + (size_t)min(b0 + u, nb - 1) * HD);
  };
  fetch(0);
  bits_t gate;
  __builtin_memcpy(&gate, p.qg + ((size_t)t * p.Hq + h) * 2 * HD + HD + PER * lane, sizeof gate);  // (as the caller has aligned it)
  float M = mb > -DM_INF ? mb : -DM_INF;
  for (int b = lane + 64; b < nb; b += 64) {
    const float m = pm[b];
    M = m > M ? m : M;
  }
  M = dm_wave_max<64>(M);
  float L = 0.f;
  chan_t O = 0.f;
  for (int b0 = 0;;) {
    const float w = dm_exp(mb - M);
#pragma unroll
    for (int s = 0; s < kMergeAhead; s += SET)
      if (b0 + s < nb)
#pragma unroll
        for (int u = s; u < s + SET; ++u) {
          const float wu = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, w), u));
          const float lu = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, lb), u));
          if (b0 + u < nb) {
            L = dm_fma(lu, wu, L);
#pragma unroll
            for (int c = 0; c < PER; ++c) O[c] = dm_fma(v[u][c], wu, O[c]);
          }
        }
    b0 += kMergeAhead;
    if (b0 >= nb) break;
    mb = pm[min(b0 + lane, nb - 1)];
    lb = pl[min(b0 + lane, nb - 1)];
    fetch(b0);
  }
  bits_t out;
#pragma unroll
  for (int c = 0; c < PER; c += 2) {
    const float g0 = dm_sigmoid_bf16(dm_bf2f_lo(gate[c / 2])), g1 = dm_sigmoid_bf16(dm_bf2f_hi(gate[c / 2]));
    out[c / 2] = dm_f2bf2(g0 * dm_rb(O[c] / L), g1 * dm_rb(O[c + 1] / L));
  }
  __builtin_memcpy(p.out + ((size_t)t * p.Hq + h) * HD + PER * lane, &out, sizeof out);
}

}  // namespace

extern "C" {

int ornith_rope_table(ornith_ctx* ctx, int npos, int dims, double theta, float* d_cos,
                      float* d_sin) {
  ORN_REQUIRE(ctx && d_cos && d_sin, "rope_table: null argument");
  ORN_REQUIRE(npos >= 1 && dims >= 2 && dims % 2 == 0 && theta > 0, "rope_table: npos=%d dims=%d",
              npos, dims);
  const int half = dims / 2;
  float* hc = (float*)malloc(sizeof(float) * (size_t)npos * half * 2);
  if (!hc) return ornith_fail(ORNITH_ERR_INVALID, "rope_table: out of host memory");
  float* hs = hc + (size_t)npos * half;
  for (int i = 0; i < half; ++i) {
    const double inv_freq = pow(theta, -(double)i / (double)half);
    for (int pos = 0; pos < npos; ++pos) {
      const double ang = (double)pos * inv_freq;
      hc[(size_t)pos * half + i] = (float)cos(ang);
      hs[(size_t)pos * half + i] = (float)sin(ang);
    }
  }
  int rc = ornith_upload(ctx, d_cos, hc, sizeof(float) * (size_t)npos * half);
  if (!rc) rc = ornith_upload(ctx, d_sin, hs, sizeof(float) * (size_t)npos * half);
  free(hc);
  return rc;
}

static int prep_args(ornith_ctx* ctx, const void* d_qg, const void* d_kx, const void* d_vx, const void* d_q_norm_w,
                     const void* d_k_norm_w, int T, int Hq, int Hkv, int hd, int rope_dims, float eps,
                     const float* d_cos, const float* d_sin, int table_npos, int offset, const int* d_offset, int cap,
                     void* d_q_rot, void* d_k_cache, void* d_v_cache, PrepArgs* out) {
  ORN_REQUIRE(ctx && d_qg && d_kx && d_vx && d_q_norm_w && d_k_norm_w && d_cos && d_sin && d_q_rot &&
                  d_k_cache && d_v_cache,
              "attn_prep: null argument");
  ORN_REQUIRE(hd == 256 || hd == 128, "attn_prep: head_dim %d (128 or 256)", hd);
  const int per = hd / 64, half = rope_dims / 2;
  ORN_REQUIRE(rope_dims >= 2 * per && rope_dims <= hd && half % per == 0 &&
                  ((half / per) & (half / per - 1)) == 0,
              "attn_prep: rope_dims=%d does not tile head_dim %d", rope_dims, hd);
  ORN_REQUIRE(T >= 1 && T <= 65535 && Hq >= 1 && Hkv >= 1 && Hq % Hkv == 0, "attn_prep: T=%d Hq=%d Hkv=%d",
              T, Hq, Hkv);
  ORN_REQUIRE(offset >= 0 && offset + T <= cap && offset + T <= table_npos,
              "attn_prep: rows [%d,%d) do not fit cache capacity %d / rope table %d", offset,
              offset + T, cap, table_npos);
  PrepArgs p{};
  p.qg = (const bf16_t*)d_qg;
  p.kx = (const bf16_t*)d_kx;
  p.vx = (const bf16_t*)d_vx;
  p.qw = (const bf16_t*)d_q_norm_w;
  p.kw = (const bf16_t*)d_k_norm_w;
  p.cos_t = d_cos;
  p.sin_t = d_sin;
  p.d_offset = d_offset;
  p.q_rot = (bf16_t*)d_q_rot;
  p.k_cache = (bf16_t*)d_k_cache;
  p.v_cache = (bf16_t*)d_v_cache;
  p.T = T;
  p.Hq = Hq;
  p.Hkv = Hkv;
  p.offset = offset;
  p.cap = cap;
  p.npos = table_npos;
  p.half = half;
  p.eps = eps;
  *out = p;
  return ORNITH_OK;
}

static int prep_launch(ornith_ctx* ctx, const PrepArgs& p, int hd) {
  dim3 grid(p.Hq + 2 * p.Hkv, p.T);
  if (hd == 256)
    hipLaunchKernelGGL(attn_prep_kernel<4>, grid, dim3(64), 0, ctx->stream, p);
  else
    hipLaunchKernelGGL(attn_prep_kernel<2>, grid, dim3(64), 0, ctx->stream, p);
  ORN_LAUNCH_CHECK("attn_prep_kernel");
  return ORNITH_OK;
}

int ornith_attn_prep(ornith_ctx* ctx, const void* d_qg, const void* d_kx, const void* d_vx,
                     const void* d_q_norm_w, const void* d_k_norm_w, int T, int Hq, int Hkv, int hd,
                     int rope_dims, float eps, const float* d_cos, const float* d_sin, int table_npos,
                     int offset, const int* d_offset, int cap, void* d_q_rot, void* d_k_cache,
                     void* d_v_cache) {
  PrepArgs p;
  int rc = prep_args(ctx, d_qg, d_kx, d_vx, d_q_norm_w, d_k_norm_w, T, Hq, Hkv, hd, rope_dims, eps, d_cos, d_sin,
                     table_npos, offset, d_offset, cap, d_q_rot, d_k_cache, d_v_cache, &p);
  if (rc) return rc;
  return prep_launch(ctx, p, hd);
}

// prep != null: the prep of the same rows has not been launched yet; it is done inside the
// attention launch where that launch's form can (the 1024-thread and eight-head forms, T <= 8, static offset), by
// its own launch first otherwise
static int sdpa_decode(ornith_ctx* ctx, const void* d_q_rot, const void* d_k_cache, const void* d_v_cache,
                       const void* d_qg, int T, int Hq, int Hkv, int hd, int offset, const int* d_offset, int cap,
                       float scale, void* d_out, const PrepArgs* prep) {
  ORN_REQUIRE(ctx && d_q_rot && d_k_cache && d_v_cache && d_qg && d_out, "sdpa_decode: null argument");
  ORN_REQUIRE(hd == 256 || hd == 128, "sdpa_decode: head_dim %d (128 or 256)", hd);
  // prompt chunks: the matrix-core kernel (outside the exact window, like the projections)
  if (T >= kPrefillRows && hd == 256 && !d_offset) {
    if (prep) {
      int rc = prep_launch(ctx, *prep, hd);
      if (rc) return rc;
    }
    return ornith_sdpa_prefill_gated(ctx, d_q_rot, d_k_cache, d_v_cache, d_qg, T, Hq, Hkv, hd, offset, cap,
                                     scale, d_out);
  }
  ORN_REQUIRE(T >= 1 && T <= 64 && Hq >= 1 && Hkv >= 1 && Hq % Hkv == 0, "sdpa_decode: T=%d Hq=%d Hkv=%d",
              T, Hq, Hkv);
  ORN_REQUIRE(offset >= 0 && offset + T <= cap, "sdpa_decode: rows [%d,%d) exceed capacity %d", offset,
              offset + T, cap);
  // with a device-side offset the grid must cover the whole cache
  const int nblk = d_offset ? (cap + ATT_KB - 1) / ATT_KB : (offset + T - 1) / ATT_KB + 1;
  const size_t per = (size_t)T * Hq * nblk;
  void* base = nullptr;
  int rc = ornith_scratch(ctx, (per * (hd + 2)) * 4 + 1024, &base);
  if (rc) return rc;
  ScratchCursor sc(base);
  SdpaArgs p{};
  p.q_rot = (const bf16_t*)d_q_rot;
  p.k_cache = (const bf16_t*)d_k_cache;
  p.v_cache = (const bf16_t*)d_v_cache;
  p.qg = (const bf16_t*)d_qg;
  p.d_offset = d_offset;
  p.part_m = sc.take<float>(per);
  p.part_l = sc.take<float>(per);
  p.part_o = sc.take<float>(per * hd);
  p.out = (bf16_t*)d_out;
  p.T = T;
  p.Hq = Hq;
  p.Hkv = Hkv;
  p.offset = offset;
  p.cap = cap;
  p.nblk = nblk;
  p.scale = scale;
  // Which form. One 1024-thread workgroup a (key block, head, row) has the shorter chain, but 150 KB of LDS
  // let a compute unit hold one of them: a round takes as long as the whole call of the many form (four
  // heads of a KV group a workgroup, two workgroups a compute unit), so it is the faster one for as long as
  // it is one round. Whole calls, us, 1024-thread form / many form, two KV groups of eight heads of 256 (with an
  // earlier merge launch, which took 1 to 1.5 more of both):
  // 256 workgroups of the first (one row at 4000 keys, four at 1000) 13.4 / 16.7, 288 (three rows at 1500)
  // 20.1 / 16.8, 384 20.3 / 16.9, 768 27.4 / 17.0, 1536 47.8 / 22.2; head width 128, 256: 11.3 / 13.0, 384: 16.8 / 13.3.
  // KV groups that are no multiple of four heads, whose last workgroup repeats heads, turn at the same
  // place: groups of six 13.2 / 16.6 at 192 and 21.4 / 16.8 at 288, of three 13.0 / 16.7 and 20.0 / 16.8, of two
  // 15.9 / 18.2 at 256 and 21.4 / 17.0 at 384, of one (four times the arithmetic) 13.4 / 16.8 at 256, level from 288
  // to 512 (20.9 / 21.7, 22.9 / 22.7), 38.3 / 31.9 at 768.
  // Inside the first key block the 1024-thread form finishes by itself, without the merge launch, and a second
  // round is still ahead: 31 rows (496 workgroups) at 0 / 200 keys 12.0 / 22.5 and 17.1 / 22.8.
  const int last_max = (d_offset ? cap - 1 : (offset + T - 1 < cap - 1 ? offset + T - 1 : cap - 1));
  const long live = (long)(last_max / ATT_KB + 1) * Hq * T;
  const bool many = live > (last_max < ATT_KB ? 2L : 1L) * ctx->compute_units;
  // How the 1024-thread form's workgroups are numbered. With the block running fastest and an odd number of blocks, every
  // head's workgroup fetches a (block, KV head) into another die's L2, the longer the more blocks there are; by die it
  // is fetched once. One row of two KV groups of eight heads, us, block fastest / by die: 5 blocks 13.9 / 12.6, 7
  // 14.8 / 12.6, 9 15.9 / 12.7, 13 18.0 / 12.8, 15 18.3 / 12.9; even numbers
  // level (12.4 to 13.3 both). At head width 128 the odd numbers took 12.0 to 13.5 where the even ones took 10.7 to 11.5. One or two blocks are too few to matter (12.2 / 12.4), and where the pairs leave a die more workgroups than it has
  // compute units (a workgroup has one to itself), its second round costs more than it saves (five rows, two blocks: 12.2 / 19.9).
  const long a_die = (long)((nblk * Hkv + kDies - 1) / kDies) * (Hq / Hkv) * T;
  p.by_die = nblk >= 3 && a_die * kDies <= ctx->compute_units;
  const dim3 grid = p.by_die ? dim3(sdpa_die_grid<1>(p)) : dim3(nblk, Hq, T);
  // one key block for every row, in the kernel form that knows how to finish: no merge launch
  p.finish = (last_max < ATT_KB && !many) ? 1 : 0;
  // Eight heads a workgroup where four make more workgroups than there are compute units and eight don't: a block's way
  // through a workgroup is longer (whole calls, us, two KV groups of eight heads of 256, four heads / eight: two rows at 6000 / 8100
  // keys, 192 / 256 workgroups of four, 16.3 / 18.3 and 16.7 / 18.7), but two workgroups that share a unit are longer still (two rows
  // at 9000 / 16000 keys, 288 / 504 workgroups of four, 22.2 / 19.3 and 23.9 / 21.0; four at 4200 / 6621 / 8100 20.9 / 18.3, 22.1 / 18.9 and
  // 22.6 / 19.0; eight at 2100 20.6 / 18.0). A second round of eights costs what it saved (four rows at 9000 / 12000 keys
  // 29.0 / 32.3 and 29.9 / 32.8, at 16000 35.0 / 33.4).
  const long pairs = (long)(last_max / ATT_KB + 1) * Hkv * T, group = Hq / Hkv;
  // (its keys go from memory to LDS, 16 bytes a lane, and its new values come 8 bytes a lane in the buffer form: rows that are not
  // aligned for that take the four-head form, and a prep launch)
  const bool eight = many && pairs * ((group + 3) / 4) > ctx->compute_units && pairs * ((group + 7) / 8) <= ctx->compute_units &&
                     (((uintptr_t)d_k_cache | (uintptr_t)d_v_cache) & 15) == 0;
  const bool fold = prep && (!many || (eight && ((uintptr_t)prep->vx & 7) == 0)) && !d_offset && T <= 8 && ornith_option_fuse_attn_prep();
  PrepArgs pq{};
  if (prep) {
    pq = *prep;
    if (!fold) {
      const int rcp = prep_launch(ctx, pq, hd);
      if (rcp) return rcp;
    }
  }
  if (eight) {
    typedef void (*Kernel)(SdpaArgs, PrepArgs);
    static const Kernel kernels[2][2] = {{sdpa_partial_eight_kernel<128, false>, sdpa_partial_eight_kernel<128, true>},
                                         {sdpa_partial_eight_kernel<256, false>, sdpa_partial_eight_kernel<256, true>}};
    const int bytes[2] = {sdpa_eight_bytes<128>(), sdpa_eight_bytes<256>()};
    if (!(ctx->lds_attr_set & 16)) {
      for (int w = 0; w < 2; ++w)
        for (const Kernel k : kernels[w])
          ORN_HIP(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, bytes[w]));
      ctx->lds_attr_set |= 16;
    }
    hipLaunchKernelGGL(kernels[hd == 256][fold], dim3(sdpa_die_grid<kEightHeads>(p)), dim3(512), bytes[hd == 256], ctx->stream, p, pq);
  } else if (many) {
    if (hd == 256)
      hipLaunchKernelGGL(sdpa_partial_many_kernel<256>, dim3(sdpa_die_grid<kManyHeads>(p)), dim3(512), 0, ctx->stream, p);
    else
      hipLaunchKernelGGL(sdpa_partial_many_kernel<128>, dim3(sdpa_die_grid<kManyHeads>(p)), dim3(512), 0, ctx->stream, p);
  } else if (hd == 256) {
    // 150 KB of LDS a block (the whole key block staged at once): asked for once per kernel
    if (!(ctx->lds_attr_set & 1)) {
      ORN_HIP(hipFuncSetAttribute((const void*)sdpa_partial_kernel<256, false>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, sdpa_stage_bytes<256>()));
      ORN_HIP(hipFuncSetAttribute((const void*)sdpa_partial_kernel<256, true>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, sdpa_stage_bytes<256>()));
      ctx->lds_attr_set |= 1;
    }
    if (fold)
      hipLaunchKernelGGL((sdpa_partial_kernel<256, true>), grid, dim3(SDPA_NT), sdpa_stage_bytes<256>(), ctx->stream, p, pq);
    else
      hipLaunchKernelGGL((sdpa_partial_kernel<256, false>), grid, dim3(SDPA_NT), sdpa_stage_bytes<256>(), ctx->stream, p, pq);
  } else {
    if (!(ctx->lds_attr_set & 2)) {
      ORN_HIP(hipFuncSetAttribute((const void*)sdpa_partial_kernel<128, false>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, sdpa_stage_bytes<128>()));
      ORN_HIP(hipFuncSetAttribute((const void*)sdpa_partial_kernel<128, true>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, sdpa_stage_bytes<128>()));
      ctx->lds_attr_set |= 2;
    }
    if (fold)
      hipLaunchKernelGGL((sdpa_partial_kernel<128, true>), grid, dim3(SDPA_NT), sdpa_stage_bytes<128>(), ctx->stream, p, pq);
    else
      hipLaunchKernelGGL((sdpa_partial_kernel<128, false>), grid, dim3(SDPA_NT), sdpa_stage_bytes<128>(), ctx->stream, p, pq);
  }
  ORN_LAUNCH_CHECK("sdpa_partial_kernel");
  if (p.finish) return ORNITH_OK;
  if (hd == 256)
    hipLaunchKernelGGL(sdpa_merge_kernel<256>, dim3(Hq, T), dim3(64), 0, ctx->stream, p);
  else
    hipLaunchKernelGGL(sdpa_merge_kernel<128>, dim3(Hq, T), dim3(64), 0, ctx->stream, p);
  ORN_LAUNCH_CHECK("sdpa_merge_kernel");
  return ORNITH_OK;
}

int ornith_sdpa_decode_gated(ornith_ctx* ctx, const void* d_q_rot, const void* d_k_cache,
                             const void* d_v_cache, const void* d_qg, int T, int Hq, int Hkv, int hd,
                             int offset, const int* d_offset, int cap, float scale, void* d_out) {
  return sdpa_decode(ctx, d_q_rot, d_k_cache, d_v_cache, d_qg, T, Hq, Hkv, hd, offset, d_offset, cap, scale, d_out,
                     nullptr);
}

int ornith_attn_decode(ornith_ctx* ctx, const void* d_qg, const void* d_kx, const void* d_vx,
                       const void* d_q_norm_w, const void* d_k_norm_w, int T, int Hq, int Hkv, int hd,
                       int rope_dims, float eps, const float* d_cos, const float* d_sin, int table_npos,
                       int offset, int cap, float scale, void* d_q_rot, void* d_k_cache, void* d_v_cache,
                       void* d_out) {
  PrepArgs p;
  int rc = prep_args(ctx, d_qg, d_kx, d_vx, d_q_norm_w, d_k_norm_w, T, Hq, Hkv, hd, rope_dims, eps, d_cos, d_sin,
                     table_npos, offset, nullptr, cap, d_q_rot, d_k_cache, d_v_cache, &p);
  if (rc) return rc;
  return sdpa_decode(ctx, d_q_rot, d_k_cache, d_v_cache, d_qg, T, Hq, Hkv, hd, offset, nullptr, cap, scale, d_out, &p);
}

}  // extern "C"
