// Pieces shared by the grouped GEMM kernels (internal to libttamd_moe.so).
#pragma once

#include <algorithm>

#include "common.h"

namespace ttamd {

// Epilogue variants of the token-row GEMMs.
enum Epi {
  EPI_STORE = 0,       // out[q][p] = acc
  EPI_SWIGLU = 1,      // gate/up pairs -> silu(clamp(gate)) * clamp(up)
  EPI_SCATTER = 2,     // out[dest[q]][p] = scale[q] * acc
  EPI_SWIGLU_BWD = 3,  // dh from dA = acc and the saved pre-activation h
};

// 1 / (1 + exp(-x)) with the hardware reciprocal (1 ulp) in place of an
// IEEE division (about ten instructions): the GEMM epilogues that use it are
// VALU-bound and round their results to bf16.
__device__ __forceinline__ float sigmoid_f(float x) { return __builtin_amdgcn_rcpf(1.f + __expf(-x)); }
__device__ __forceinline__ float silu_f(float x) { return x * sigmoid_f(x); }

// torch.clamp(x, max=L) and torch.clamp(x, -L, L): NaN stays NaN (the IEEE
// 754-2019 minimum / maximum, v_minimum3_f32 / v_maximum3_f32 on gfx950),
// where fminf / fmaxf would return the limit.
__device__ __forceinline__ float clamp_max_nan(float x, float L) { return __builtin_elementwise_minimum(x, L); }
__device__ __forceinline__ float clamp_nan(float x, float L) {
  return __builtin_elementwise_maximum(__builtin_elementwise_minimum(x, L), -L);
}

// Token-row tiles: table[i] = {expert, first row, end row, 0}, at most
// kFwdTileRows rows (bf16 forward and dgrad) or kFp8TileRows (fp8).  The
// workspace is sized for tiles of kTileRows rows, fewer rows than either,
// so it always holds the table.
constexpr int kTileRows = 128;
constexpr int kFwdTileRows = 320;

// Tile plan of a token-row GEMM: int4 header {number of tiles, number of
// small tiles, ...}, the arrival counters of the split tail tiles
// (kSplitTiles ints, zeroed whenever a table is built and left at zero by
// every GEMM that uses them), the tile table, then the table of the
// small-tile kernel (filled where small_tile_rows(M, E) > 0; the room for it
// is there for every M).
constexpr int kSplitTiles = 512;
struct TileTable {
  int* count;
  int* split_cnt;
  int4* table;
  int small_rows;  // largest small tile, 0: no small table
  int* small_count;
  int4* small_table;
};

inline int max_row_tiles(int M, int E) { return M / kTileRows + E + 1; }

// Small-tile kernel (gemm_small.hip): token tiles of small_tile_rows(M, E)
// rows at most, 128 or 256 weight rows.  Whether a GEMM of a plan takes it,
// and with how many weight rows, is small_tile_cols' choice (gemm.hip); the
// table exists wherever it could be chosen.  64-row tiles for experts that
// mostly fit one, and for few rows in all (one expert of 2048 x 4096, 200 rows
// 30 us against 39 with 128-row tiles; of 5120 x 8192, 320 rows 59 against 75,
// 640 rows 80 against 83).  Near the line it goes either way: one of 7168 x
// 2048, 640 rows 45 against 33; one of 2048 x 768, 800 rows 10 against 12.
constexpr int kSmallAvgRows = 100;
constexpr int kSmallMaxRows = 8192;
inline int64_t small_rows64_max(int E) { return std::max<int64_t>(32 * (int64_t)E + 31, 768); }
inline int64_t small_rows128_max(int E) { return std::max<int64_t>(kSmallAvgRows * (int64_t)E, kSmallMaxRows); }
inline int small_tile_rows(int M, int E) {
  if (M <= small_rows64_max(E)) return 64;
  return M <= small_rows128_max(E) ? 128 : 0;
}
// An expert's c rows make at most ceil(c / rows) tiles.
inline int max_small_tiles(int M, int E) {
  const int rows = small_tile_rows(M, E);
  return rows > 0 ? M / rows + E + 1 : 0;
}
// The most small tiles of any call of at most M rows: what a plan has room
// for, so that one sized for the largest batch serves every smaller one.
inline int64_t small_table_tiles(int64_t M, int E) {
  return std::max(std::min(M, small_rows64_max(E)) / 64, std::min(M, small_rows128_max(E)) / 128) + E + 1;
}

inline TileTable tile_table_in(void* ws, int M, int E) {
  TileTable t;
  t.count = (int*)ws;
  t.split_cnt = (int*)ws + 4;
  t.table = (int4*)(t.split_cnt + kSplitTiles);
  t.small_rows = small_tile_rows(M, E);
  t.small_count = t.count + 1;
  t.small_table = t.table + max_row_tiles(M, E);
  return t;
}

// Tail split of the forward / dgrad GEMM: the tiles left over after the
// last full round of the persistent walk are cut along k into pieces that
// run on the otherwise idle CUs; each piece writes its fp32 accumulators
// (kSplitPartBytes, register order) to the partial-sum area of the GEMM's
// workspace, and the last piece of a tile to arrive adds them in piece
// order and runs the epilogue.  At most kSplitMaxPieces pieces per tile,
// each of at least kSplitMinStages k stages, and only for walks of at most
// kSplitMaxRounds full rounds: with more, the ragged tile heights of skewed
// routing decide the finish time more than the leftover tiles do (C4's
// Zipf w13, 7 rounds + 32 tiles: no gain; C3's shared w13, 6 rounds + 128
// tiles of equal height: -40 us).
constexpr size_t kSplitPartBytes = 327680;  // 8 waves x 160 fp32 x 64 lanes
constexpr int kSplitMaxPieces = 8;
constexpr int kSplitMinStages = 8;
constexpr int kSplitMaxRounds = 6;
// Pieces per leftover tile of a walk of R full rounds of G workgroups and rt
// leftover tiles (1: no split).  The last piece reads every partial, so at
// most sqrt(ksteps / 2) pieces, and two only for long reductions.
__host__ __device__ inline int split_pieces(int R, int rt, int G, int ksteps, int most) {
  if (rt <= 0 || rt > kSplitTiles || R > kSplitMaxRounds) return 1;
  int np = std::max(1, std::min(std::min(G / rt, most), ksteps / kSplitMinStages));
  while (np > 1 && ksteps < 2 * np * np) --np;
  return np == 2 && ksteps < 64 ? 1 : np;
}

// Height of the tiles of an expert's c > 0 rows, and their number.
__host__ __device__ inline int tile_height(int c, int max_rows) {
  const int n = (c + max_rows - 1) / max_rows;
  return (((c + n - 1) / n) + 31) & ~31;
}
inline int tiles_of(int c, int max_rows) { return c > 0 ? (c + tile_height(c, max_rows) - 1) / tile_height(c, max_rows) : 0; }

// Builds one tile table with one workgroup of NT threads (every thread
// calls it; it synchronises the workgroup).  `range(e, r0, r1)` gives the
// rows [r0, r1) of expert e.  An expert's rows are split into the fewest
// tiles of at most max_rows rows, of equal height rounded up to 32 rows
// (540 rows at max_rows = 320 give 2 tiles of 288 rather than 320 + 220);
// tiles are numbered in expert order.  Entries past the last tile, up to
// max_tiles, are {-1, 0, 0, 0}.  sh: NT / 64 + 1 ints of LDS.
template <int NT, typename Range>
__device__ void block_tile_table(Range range, int E, int max_tiles, int max_rows, int4* __restrict__ table,
                                 int* __restrict__ count, int* sh) {
  constexpr int NW = NT / kWave;
  const int tid = threadIdx.x;
  const int w = tid / kWave, l = lane_id();
  int carry = 0;
  for (int e0 = 0; e0 < E; e0 += NT) {
    const int e = e0 + tid;
    int r0 = 0, r1 = 0, nt = 0, h = max_rows;
    if (e < E) {
      range(e, r0, r1);
      const int c = r1 - r0;
      if (c > 0) {
        h = tile_height(c, max_rows);
        nt = (c + h - 1) / h;
      }
    }
    const int incl = wave_inclusive_scan(nt);
    if (l == kWave - 1) sh[w] = incl;
    __syncthreads();
    if (w == 0) {
      const int v = (l < NW) ? sh[l] : 0;
      const int vi = wave_inclusive_scan(v);
      if (l < NW) sh[l] = vi;  // inclusive over waves
    }
    __syncthreads();
    const int start = carry + ((w > 0) ? sh[w - 1] : 0) + incl - nt;
    for (int t = 0; t < nt; ++t) {
      const int i = start + t;
      if (i < max_tiles) table[i] = make_int4(e, r0 + t * h, min(r0 + (t + 1) * h, r1), 0);
    }
    carry += sh[NW - 1];
    __syncthreads();  // sh is rewritten by the next round
  }
  for (int i = carry + tid; i < max_tiles; i += NT) table[i] = make_int4(-1, 0, 0, 0);
  if (tid == 0) *count = min(carry, max_tiles);
}

// The whole plan: both tables (the small one where it exists) and zeroed
// split-tile arrival counters.
template <int NT, typename Range>
__device__ void block_tile_plan(Range range, int E, int max_tiles, int max_rows, const TileTable& t,
                                int max_small, int* sh) {
  for (int i = threadIdx.x; i < kSplitTiles; i += NT) t.split_cnt[i] = 0;
  block_tile_table<NT>(range, E, max_tiles, max_rows, t.table, t.count, sh);
  if (max_small > 0) block_tile_table<NT>(range, E, max_small, t.small_rows, t.small_table, t.small_count, sh);
}

// Forward GEMM description (gemm_fwd.hip, gemm_small.hip).
//   act [M][kred] bf16, w [E][N or 2N][kred] bf16.
//   EPI_SWIGLU: n = H (w holds 2H rows: gate then up), out [M][H], h_out [M][2H].
//   EPI_STORE / EPI_SCATTER: n = N, out [M or n_dest][N].
struct FwdGemm {
  const void* act;
  const int* act_index;  // nullable: gathered activation rows (act row = act_index[j] / act_div)
  int act_div;
  int n_act;
  const void* w;
  int kred;
  int n;
  const int4* table;
  const int* n_qtiles;
  int* split_cnt;  // the plan's arrival counters
  float* part;     // nullable: partial sums of split tail tiles (no split when null)
  void* out;
  float limit;
  void* h_out;
  const float* row_scale;
  const int* dest;
  int n_dest;
  int accumulate;     // EPI_SCATTER: out[dest] = bf16(out[dest] + v) instead of bf16(v)
  int scale_sigmoid;  // EPI_SCATTER: the row scale is sigmoid(row_scale[j])
};

// Kernel arguments of the forward and dgrad GEMMs (gemm_fwd.hip).
struct FwdArgs {
  const bf16_t* q;  // activations [M][kred], or [n_q_in][kred] gathered through q_index
  int64_t ldq;
  const int* q_index;  // nullable: token row j reads q row q_index[j] / q_div
  int q_div;
  int n_q_in;
  const bf16_t* p;  // weights, expert e at p + e * p_estride, rows of ldp
  int64_t p_estride;
  int64_t ldp;
  int kred;
  int n_p;       // valid weight rows (SWIGLU: H, the gate half)
  int np_tiles;  // weight-row tiles per token tile
  const int4* table;
  const int* n_qtiles;
  // tail split (null part: none); part and split_cnt adjacent (the kernel
  // reads both with one scalar load)
  float* part;
  int* split_cnt;
  int split_max;
  bf16_t* out;
  int64_t ldo;
  // EPI_SWIGLU
  int64_t hidden;
  float limit;  // NaN = no clamp
  bf16_t* h_out;
  int64_t ldh;
  // EPI_SWIGLU_BWD
  const bf16_t* h_in;  // saved pre-activation [M][2H]
  bf16_t* a_out;       // recomputed activation [M][H] (nullable)
  // EPI_SCATTER
  const float* row_scale;
  const int* dest;
  int n_dest;
  int accumulate;
  int scale_sigmoid;
};
// The split path of the forward kernel reads part and split_cnt with one
// 16-byte scalar load at offsetof(FwdArgs, part).
static_assert(offsetof(FwdArgs, split_cnt) == offsetof(FwdArgs, part) + sizeof(float*) &&
                  offsetof(FwdArgs, part) % 8 == 0,
              "FwdArgs: split_cnt must directly follow part");

// Grouped dgrad through the forward kernel's reduction-major weight mode:
// out[m, k] = sum_n dy[m, n] w[e(m), n, k], w [E, n_red, n_out].
struct DgradGemm {
  const void* dy;  // [M][n_red]
  const void* w;
  int n_red;
  int n_out;
  const int4* table;
  const int* n_qtiles;
  int* split_cnt;
  float* part;  // nullable
  void* out;  // EPI_STORE: [M][n_out]; EPI_SWIGLU_BWD: dh [M][2 n_out]
  // EPI_SWIGLU_BWD
  const void* h;  // [M][2 n_out]
  float limit;
  void* a_out;
};

// Grouped weight gradient (gemm_wgrad.hip): dw[e][n][k] = sum over the
// expert's rows m of dy[m][n] * x[m][k].
struct WgradDmaArgs {
  const bf16_t* dy;  // [M][N]
  int64_t lddy;
  const bf16_t* x;  // [M][K]
  int64_t ldx;
  const int* offs;  // inclusive, [E]
  int E, M, N, K;
  int n_tiles, k_tiles;  // per expert, 256-wide
  void* dw;              // [E][N][K]
  int dw_fp32;
  // Tail split (split_np > 1): the tiles left over after the last full
  // round are cut along the reduction rows into split_np pieces; each
  // piece writes its fp32 sums (kSplitPartBytes at most) to `part` and
  // counts its arrival in split_cnt[leftover tile] (zero on entry, left at
  // zero).  split_np <= 1: no split.
  float* part;
  int* split_cnt;
  int split_np;
};
hipError_t launch_wgrad_dma(const WgradDmaArgs& a, hipStream_t stream);
hipError_t launch_split_cnt_zero(int* split_cnt, int n, hipStream_t stream);

// Kernel arguments of the fp8 forward GEMM (gemm_fp8.hip).  Activations and
// weights are e4m3 bytes; strides are in bytes for them, in elements for
// the scale and output arrays.
struct Fp8Args {
  const uint8_t* q;  // activations [M][kred] e4m3
  int64_t ldq;
  const uint8_t* p;  // weights, expert e at p + e * p_estride, rows of ldp bytes
  int64_t p_estride;
  int64_t ldp;
  int kred;
  int np_tiles;  // weight-row tiles per token tile
  int n_p;       // weight rows N (STORE, SCATTER: the last tile may hold only 128)
  const int4* table;
  const int* n_qtiles;
  const float* sx;  // activation scales [kred/128][ldsx] (k-block major)
  int64_t ldsx;
  const float* sw;  // weight block scales, expert e at sw + e * sw_estride: [N/128][kred/128]
  int64_t sw_estride;
  bf16_t* out;
  int64_t ldo;
  // EPI_SWIGLU
  int64_t hidden;
  float limit;  // NaN = no clamp
  bf16_t* h_out;
  int64_t ldh;
  // EPI_SCATTER
  const float* row_scale;
  const int* dest;
  int n_dest;
};

// Token tiles of the fp8 GEMM have at most this many rows.
constexpr int kFp8TileRows = 256;

// Estimated time of one round of fp8 tiles of h token rows (0.01 us, k in
// stages of 128): large tiles, and the small ones' share that grows with the
// rows (on top of a time that depends on their form, fp8_choice in gemm.hip).
// `stream`: the weights stream from HBM, and a stage waits for its rows.
__host__ __device__ inline int fp8_large_round(int stages, bool stream, int h) {
  const int waits = stream ? 60 + stages * 163 + h * (820 + 5 * stages) / 100 : 450 + 463 * h / 100 + stages * 97;
  return std::max(waits, 300 + 463 * h / 100 + stages * 164 * h / 256);
}
__host__ __device__ inline int fp8_small_rows(int stages, int cols, int h) { return h * (385 + 9 * stages) * (cols / 128) / 100; }

// Small (128-row) or large fp8 tiles by their rounds of G workgroups and the
// time of a round of either.  The counts of tiles decide it, so it is made
// where they are known, on the device: the rows per expert alone do not say
// how a skewed load falls into rounds.  DeepSeek-V3 shard w13 (7168 -> 2 x
// 2048, 16 weight tiles), us, small against large: 2300 rows over 32 experts
// even 175 against 202 (2 rounds of both), Zipf(1.2) over 28 of them 247
// against 196 (38 small token tiles, 3 rounds; 32 large, 2), 3199 rows
// Zipf(1.2) over 28 248 against 280 (3 rounds of both), 3200 rows on 4 experts
// 156 against 93.  Chosen by the average rows, the small side always ran.
struct Fp8Pick {
  const int4* small_table;
  const int* small_count;
  int small_np;    // weight-row tiles per small token tile
  int small_cols;  // their weight rows
  int small_time;  // one round of small tiles without fp8_small_rows
  int rows;        // M
  int stream;      // weights stream from HBM
};
__host__ __device__ inline bool fp8_pick_small(const Fp8Pick& p, int ns, int nl, int large_np, int stages, int G) {
  // rounds of G tiles in units of 1 / 2G: after a full round, a last one of a
  // share f takes (1 + f) / 2 of it (33 small tiles, 2.06 rounds, 221 us, 47,
  // 2.94 rounds, 252; 32, 2 rounds, 171); within 7 % the small side stays
  auto rounds = [&](int tiles) {
    const int rest = tiles % G;
    return (float)(tiles < G ? 2 * G : 2 * (tiles - rest) + (rest ? G + rest : 0));
  };
  const int small = p.small_time + fp8_small_rows(stages, p.small_cols, p.rows / std::max(ns, 1));
  const int large = fp8_large_round(stages, p.stream != 0, p.rows / std::max(nl, 1));
  return rounds(ns * p.small_np) * (float)(100 * small) <= rounds(nl * large_np) * (float)(107 * large);
}

int num_cus();

// with_small: also the small-tile table, where small_tile_rows(M, E) > 0.
hipError_t launch_tile_map(const int* offs, int E, int M, int max_rows, void* ws, bool with_small,
                           hipStream_t stream);
// Forward GEMM over a tile table of at most kFwdTileRows rows per tile
// (small_cols == 0), or of at most small_rows rows and with small_cols
// weight rows per tile (gemm_small.hip).
hipError_t launch_fwd_gemm(int epi, const FwdGemm& g, int small_rows, int small_cols, hipStream_t stream);
hipError_t launch_small_gemm(int epi, FwdArgs a, int tile_rows, int tile_cols, hipStream_t stream);
// Most pieces of a split leftover tile.
int split_max();
// dgrad GEMM (EPI_STORE or EPI_SWIGLU_BWD) over the same tile table.
hipError_t launch_dgrad_gemm(int epi, const DgradGemm& g, hipStream_t stream);
// fp8 forward GEMM (gemm_fp8.hip).  rows 64: small tiles of 64 token rows x
// `cols` weight rows, whose table is a.table; rows 128: small tiles of 128 x
// `cols` (p) or the large ones (a), chosen on the device; 256: the large ones.
hipError_t launch_fp8_gemm(int epi, const Fp8Args& a, const Fp8Pick& p, int rows, int cols, hipStream_t stream);

}  // namespace ttamd
