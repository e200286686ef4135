// The few-row GEMM (mm_narrow.h) over Q4_K / Q6_K weights, and the launch rules of both families.
#include <algorithm>

#include "mm_narrow_host.h"

namespace nmm {
constexpr int kq_waves(int kind, int rows) { return rows == 16 ? (kind == kQ4K ? 5 : 4) : rows == 32 ? (kind == kQ4K ? 4 : 3) : 2; }
NMM_KERNELS(kq, false, kQ4K, kQ6K, kq_waves, 4u, nullptr, nullptr)

namespace {

int kind_of(const ornith_linear& w) {
  switch (w.mode) {
    case ORNITH_LIN_KQUANT: return w.km.kind == ORNITH_Q4K ? kQ4K : w.km.kind == ORNITH_Q6K ? kQ6K : -1;
    case ORNITH_LIN_AFFINE4: return kA4;
    case ORNITH_LIN_AFFINE8: return kA8;
    default: return -1;
  }
}
int kind_of(const ornith_kmatrix& w) {
  return w.kind == ORNITH_Q4K ? kQ4K : w.kind == ORNITH_Q6K ? kQ6K : w.kind == ORNITH_AFFINE4_G32 ? kA4 : -1;
}
bool affine(int kind) { return kind >= kA4; }

Mat mat_of(const ornith_linear& w, void* y) {
  if (w.mode == ORNITH_LIN_KQUANT)
    return {(const uint8_t*)w.km.d_qs, (const uint8_t*)w.km.d_scales, (const uint8_t*)w.km.d_dm, (bf16_t*)y, w.O, kind_of(w), 0};
  return {(const uint8_t*)w.d_w, (const uint8_t*)w.d_scales, (const uint8_t*)w.d_biases, (bf16_t*)y, w.O, kind_of(w), 0};
}
Mat mat_of(const ornith_kmatrix& w, void* y) {
  return {(const uint8_t*)w.d_qs, (const uint8_t*)w.d_scales, (const uint8_t*)w.d_dm, (bf16_t*)y, w.O, kind_of(w), 0};
}
// the kernels' 16-byte loads (the scales of 16 rows, or of what is left of the matrix, are whole
// 16-byte pieces) and 32-bit offsets inside one matrix
bool reachable(const Mat& m, int K) {
  return m.kind >= 0 && m.O >= 1 && m.q && m.s && m.d && (size_t)m.O * K < (size_t(1) << 32) && m.O * (size_t)(K / 256) % 8 == 0 &&
         (((uintptr_t)m.q | (uintptr_t)m.s | (uintptr_t)m.d) & 15) == 0 && ((uintptr_t)m.y & 7) == 0;
}
// LDS of a plain launch: activations and scales (of the widest format), or the partial tiles
int lds_bytes(const Args& a, int cols, int rows, int ct, int nw) {
  int scales = 0;
  for (int i = 0; i < a.n; ++i) {
    const int k = a.m[i].kind;
    scales = std::max(scales, k == kA4 ? nw * 4096 : cols * (a.K / 256) * (s_bytes(k) + d_bytes(k)));
  }
  return std::max(x_bytes(rows, nw) + scales, red_bytes(rows, ct, nw));
}
// wavefronts of NW that split K: as many as there are 256-wide blocks, a power of two
int k_split(int K, int nw) {
  int ks = 1;
  while (2 * ks <= nw && 2 * ks <= K / 256) ks *= 2;
  return ks;
}

}  // namespace

bool plain_ok(const ornith_linear* const* ws, int n, const void* d_x, int M, void* const* d_ys) {
  if (n < 1 || n > 4 || M < kPrefillRows || ((uintptr_t)d_x & 15) != 0) return false;
  const int K = ws[0]->K;
  if (K < 512 || K % 256 != 0 || (size_t)M * K * 2 >= (size_t(1) << 32)) return false;
  for (int i = 0; i < n; ++i) {
    const Mat m = mat_of(*ws[i], d_ys[i]);
    if (!reachable(m, K) || ws[i]->K != K || affine(m.kind) != affine(kind_of(*ws[0]))) return false;
    if (ws[i]->mode == ORNITH_LIN_KQUANT && (ws[i]->km.E != 1 || ws[i]->km.O != ws[i]->O || ws[i]->km.K != K)) return false;
  }
  if (K > 4096) return false;  // (the scales of a workgroup's rows would not fit beside the activations)
  if (affine(kind_of(*ws[0]))) return true;  // (no wider kernels)
  for (int i = 0; i < n; ++i)
    if (M > kq_rows(ws[i]->km.kind == ORNITH_Q4K, ws[i]->O, K)) return false;
  return true;
}

namespace {
// the form of one matrix, whatever shares its launch
bool tall(const ornith_linear& w, int M) { return affine(kind_of(w)) && w.O > 2048 && M > kTallFromAffine; }

int launch_tall(ornith_ctx* ctx, Args& a) {
  int kind = a.m[0].kind, lds = 0;
  a.blocks = 0;
  for (int i = 0; i < a.n; ++i) {
    a.m[i].cb0 = a.blocks;
    a.blocks += (a.m[i].O + 127) / 128;
    lds = std::max(lds, owned_lds(64, a.m[i].kind, kTall, a.K / 256));
    if (a.m[i].kind != kind) kind = -1;
  }
  a.tiles_max = (a.M + 63) / 64;
  const dim3 grid((unsigned)((a.blocks + 7) / 8 * 8 * a.tiles_max + (a.d.wgs + 7) / 8 * 8));
  return launch_affine(ctx, a, kTall, 0, 64, kind, grid, lds);
}

int launch_split(ornith_ctx* ctx, Args& a) {
  a.ks = k_split(a.K, 4);
  // The tile, columns x rows; sums and their order are the same in all of them.
  // While one workgroup a compute unit covers the product with 32-row tiles, those: a workgroup asks for its rows'
  // activations over all of K (64 rows of K = 4096: 512 KB, 4 us of the unit's address path), and half the
  // rows are half of that. us, 64-row tiles / 32-row ones: 2048 x 4096 Q4_K 51 rows 9.4 / 7.2, Q6_K 11.0 / 8.8, 4-bit affine
  // 12.6 / 9.5; 256 x 2048 Q6_K 51 .. 450 rows 6.6 .. 6.8 / 5.4 .. 5.7, 8-bit affine 7.6 / 6.4. One workgroup more and the second round
  // costs what that gave (2048 x 4096 at 100 rows 10.3 / 10.3, at 150 14.3 / 14.7; 256 x 2048 8-bit affine at 600 7.8 / 10.5).
  // With 32 columns the same holds from four blocks a wavefront on (2048 x 4096 at 100 rows: Q4_K 10.3 / 9.3, 4-bit affine 12.1 / 11.2;
  // K = 2048 has two: 256 columns at 600 rows 7.2 / 7.6, 8-bit affine 7.9 / 9.0), but for Q6_K, whose unpacking is the longer
  // part (80 / 100 / 128 rows 10.7 / 11.5 / 12.8, here 12.1 / 12.2 / 12.2).
  // With 64-row tiles 64 columns (four tiles a wavefront, each activation fragment used four times) once that gives
  // most compute units a workgroup, else 32 or 16. They have to share a compute unit once there is more than one for each: with
  // Q6_K's 18 bytes of scales a block they don't at K = 4096 (82 KB of LDS), and take 32 columns (2048 columns, 600 / 700 / 900 rows
  // 45.7 / 46.2 / 46.3 -> 35.4 / 36.0 / 45.1; at 450 rows, one each, 24.1 / 24.8).
  auto blocks_of = [&](int ct) {
    const int cols = (4 / a.ks) * ct * 16;
    a.blocks = 0;
    for (int i = 0; i < a.n; ++i) {
      a.m[i].cb0 = a.blocks;
      a.blocks += (a.m[i].O + cols - 1) / cols;
    }
    return a.blocks;
  };
  bool q6 = false;
  for (int i = 0; i < a.n; ++i) q6 = q6 || a.m[i].kind == kQ6K;
  const int units = ctx->compute_units, thirty = (a.M + 31) / 32, sixty = (a.M + 63) / 64;
  int ct = 4, rows = 64;
  if ((long)blocks_of(1) * thirty <= units) {
    ct = 1;
    rows = 32;
  } else if (!q6 && a.K >= 4096 && (long)blocks_of(2) * thirty <= units) {
    ct = 2;
    rows = 32;
  } else {
    auto suits = [&]() {
      const long n = (long)blocks_of(ct) * sixty;
      return n >= 3 * units / 4 && (n <= units || lds_bytes(a, (4 / a.ks) * ct * 16, 64, ct, 4) <= kLdsBytes / 2);
    };
    while (ct > 1 && !suits()) ct /= 2;
  }
  const int row_tiles = rows == 32 ? thirty : sixty;
  const dim3 grid(blocks_of(ct) + (a.d.wgs + row_tiles - 1) / row_tiles, row_tiles);
  const int lds = lds_bytes(a, (4 / a.ks) * ct * 16, rows, ct, 4);
  return affine(a.m[0].kind) ? launch_affine(ctx, a, kPlain, ct, rows, -1, grid, lds) : launch_kq(ctx, a, kPlain, ct, rows, -1, grid, lds);
}
}  // namespace

// A riding tile is a workgroup of one 16 x 16 tile, which asks for 3.2 times what a tile of the dense launch's four-tile form does: riding
// saves that launch (4 to 6 us) and loses on large products. us, beside 4096 x 2048 of Q4_K, a launch of its own / riding (tiles): up to
// 192 rows, where the launch of its own is a chain whatever its width, 1024 columns, 128 rows 20.0 / 15.5 (512), 192 rows 25.4 / 21.4 (768); 2048
// columns, 96 rows 23.5 / 21.2 (768), 192 36.2 / 31.8 (1536); 4096 columns, 128 rows 40.5 / 37.8 (2048), 192 48.6 / 54.1 (3072). More rows: 256
// columns, 448 rows 28.2 / 24.9 (448), 600 36.8 / 31.3 (608), 900 38.1 / 42.4 (912); 512 columns, 320 rows 30.4 / 31.0 (640), 448 30.6 / 34.7 (896);
// 2048 columns, 320 rows 50.4 / 52.6, 900 107 / 128 (7296). Over 4-bit affine weights alike; the a / b heads (64 columns) beside 12288 x 2048 of
// them: 600 rows 68.5 / 65.4 (152), 2500 242 / 237 (628), 4096 382.1 / 382.2 (1024), 8192 755 / 757 (2048).
bool riders_ok(ornith_ctx* ctx, const ornith_linear* const* ws, int n, int K, int M) {
  long tiles = 0;
  for (int i = 0; i < n; ++i) {
    if (ws[i]->mode != ORNITH_LIN_DENSE || !ws[i]->d_w || ws[i]->K != K || ws[i]->O < 1 || ((uintptr_t)ws[i]->d_w & 15) != 0) return false;
    tiles += (ws[i]->O + 15) / 16;
  }
  return n >= 1 && n <= 2 && K % 2048 == 0 && 2 * tiles * ((M + 15) / 16) <= (M <= 192 ? 16L : 5L) * ctx->compute_units;
}

int plain(ornith_ctx* ctx, const ornith_linear* const* ws, int n, const void* d_x, int M, void* const* d_ys,
          const ornith_linear* const* riders, int n_riders, void* const* d_yr) {
  Riders d{};
  for (int i = 0; i < n_riders; ++i) {
    d.w[i] = (const bf16_t*)riders[i]->d_w;
    d.y[i] = (bf16_t*)d_yr[i];
    d.O[i] = riders[i]->O;
    d.tiles += (riders[i]->O + 15) / 16;
  }
  d.wgs = (M + 15) / 16 * d.tiles;
  // the matrices of one form share a launch; the riders go with the first
  for (const bool form : {true, false}) {
    Args a{};
    a.x = (const bf16_t*)d_x;
    a.M = M;
    a.K = ws[0]->K;
    for (int i = 0; i < n; ++i)
      if (tall(*ws[i], M) == form) a.m[a.n++] = mat_of(*ws[i], d_ys[i]);
    if (a.n == 0) continue;
    a.d = d;
    d = Riders{};
    const int rc = form ? launch_tall(ctx, a) : launch_split(ctx, a);
    if (rc) return rc;
  }
  return ORNITH_OK;
}

int tile_rows(int pairs, int E) {
  // The smallest tile that most experts' shares of the pairs fit (an expert over it takes a second
  // tile and has its weights unpacked twice): one standard deviation to spare. Smaller tiles keep
  // more wavefronts on a compute unit, which pays for the few that spill over (5600 pairs of 256
  // experts, gate and up / down: 64-row tiles 134 / 88 us, 32-row ones 113 / 77).
  const int avg = (pairs + E - 1) / E;
  int spare = 0;
  while (spare * spare < avg) ++spare;
  return avg + spare <= 16 ? 16 : avg + spare <= 32 ? 32 : 64;
}

bool experts_ok(const ornith_kmatrix* w, const void* d_x, size_t x_rows, const void* d_y) {
  return w->K >= 512 && w->K <= 4096 && w->K % 256 == 0 && w->E <= 1024 && ((uintptr_t)d_x & 15) == 0 &&
         x_rows * w->K * 2 < (size_t(1) << 32) && reachable(mat_of(*w, const_cast<void*>(d_y)), w->K);
}

namespace {
int launch_gathered(ornith_ctx* ctx, Args& a, int mode, const Plan& p, int O) {
  a.pair = p.pair;
  a.tile_expert = p.tile_expert;
  a.tile_start = p.tile_start;
  a.tile_count = p.tile_count;
  a.n_tiles = p.n_tiles;
  a.tiles_max = (int)p.tiles_max;
  a.up_magic = dm_div_magic(a.up_div);
  const int halves = mode == kGateUp ? 2 : 1, cols = 128 / halves;
  a.blocks = (O + cols - 1) / cols;
  // LDS: activations, and the scales of the workgroup's 128 rows
  int kind = a.m[0].kind, lds = 0;
  for (int i = 0; i < 4; ++i) {
    if (!a.m[i].q) continue;
    const int k = a.m[i].kind;
    lds = std::max(lds, owned_lds(p.rows, k, mode, a.K / 256));
    if (k != kind) kind = -1;
  }
  const dim3 grid((unsigned)(a.blocks * ((p.tiles_max + 7) / 8 * 8)));
  return affine(a.m[0].kind) ? launch_affine(ctx, a, mode, 0, p.rows, kind, grid, lds)
                             : launch_kq(ctx, a, mode, 0, p.rows, kind, grid, lds);
}
}  // namespace

int gathered(ornith_ctx* ctx, const ornith_kmatrix* w, const ornith_linear* shared, const void* d_x, int pairs, int up_div,
             const Plan& p, void* d_y) {
  Args a{};
  a.m[0] = mat_of(*w, d_y);
  if (shared) a.m[2] = mat_of(*shared, d_y);
  a.x = (const bf16_t*)d_x;
  a.M = pairs;
  a.K = w->K;
  a.up_div = up_div;
  a.pairs = pairs;
  a.E = w->E;
  return launch_gathered(ctx, a, kGather, p, w->O);
}

int gate_up(ornith_ctx* ctx, const ornith_moe_weights* w, const void* d_x, int pairs, const Plan& p, void* d_act) {
  Args a{};
  a.m[0] = mat_of(w->ex_gate, d_act);
  a.m[1] = mat_of(w->ex_up, d_act);
  a.m[2] = mat_of(w->sh_gate, d_act);
  a.m[3] = mat_of(w->sh_up, d_act);
  a.x = (const bf16_t*)d_x;
  a.M = pairs;
  a.K = w->ex_gate.K;
  a.up_div = w->top_k;
  a.pairs = pairs;
  a.E = w->ex_gate.E;
  return launch_gathered(ctx, a, kGateUp, p, w->ex_gate.O);
}

bool moe_ok(const ornith_moe_weights* w, const void* d_x, int T, const void* d_act, const void* d_y) {
  if (w->ex_dense) return false;
  const int pairs = T * w->top_k, E = w->ex_gate.E, H = w->router.K;
  const int kg = kind_of(w->ex_gate), sg = kind_of(w->sh_gate);
  if (kg < 0 || sg < 0 || kind_of(w->ex_up) != kg || kind_of(w->sh_up) != sg || w->sh_gate.O != w->ex_gate.O) return false;
  if (affine(kg) != affine(sg) || affine(kind_of(w->ex_down)) != affine(kg) || affine(kind_of(w->sh_down)) != affine(kg)) return false;
  if (!experts_ok(&w->ex_gate, d_x, T, d_act) || !experts_ok(&w->ex_up, d_x, T, d_act) ||
      !experts_ok(&w->ex_down, d_act, (size_t)pairs + T, d_y))
    return false;
  const ornith_linear* sh[3] = {&w->sh_gate, &w->sh_up, &w->sh_down};
  for (int i = 0; i < 3; ++i) {
    if (!reachable(mat_of(*sh[i], const_cast<void*>(i < 2 ? d_act : d_y)), sh[i]->K)) return false;
    if (sh[i]->mode == ORNITH_LIN_KQUANT && (sh[i]->km.O != sh[i]->O || sh[i]->km.K != sh[i]->K || sh[i]->km.E != 1)) return false;
  }
  if (w->ex_gate.O % 4 != 0 || H % 4 != 0) return false;
  // experts with many rows belong to the tall tiles of kq_mm.hip; the affine format has none
  return affine(kg) || pairs < kNarrowPairs * E;
}

}  // namespace nmm
