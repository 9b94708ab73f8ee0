// Host-side launchers of the grouped GEMMs and the device tile scheduler.
//
// The GEMM kernels live in gemm_fwd.hip (forward, dgrad), gemm_wgrad.hip
// (weight gradient) and gemm_fp8.hip (fp8 forward); this file builds the
// token-row tile table on the device (no count reaches the host) and maps
// each C-ABI operation onto a kernel configuration.
//
// Reference semantics (torchtitanturbo/models/common/npu_gmm.py):
//   :17-18, :31, :38  torch._grouped_mm(x, w.transpose(-2, -1), offs)
//   :32-36            optional clamp with swiglu_limit
//   :37               npu_swiglu: silu(gate) * up, gate = first H columns
#include <algorithm>

#include "common.h"
#include "gemm_common.h"
#include "kernels.h"

namespace ttamd {

// ---------------------------------------------------------------------------
// Tile table: token tile i -> {expert, first row, end row}.  Built on the
// device from the inclusive group offsets, so no count reaches the host
// (block_tile_table: equal-height tiles of at most max_rows rows per
// expert).  A null offs means one expert (E == 1) with all M rows.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(1024) void tile_map_kernel(const int* __restrict__ offs, int E,
                                                        int M, int max_tiles, int max_rows,
                                                        const TileTable t, int max_small) {
  __shared__ int sh[1024 / kWave + 1];
  auto range = [&](int e, int& r0, int& r1) {
    // offs == nullptr: one expert owning all M rows
    const int a = (e == 0 || !offs) ? 0 : offs[e - 1];
    const int b = offs ? offs[e] : M;
    r0 = min(max(a, 0), M);
    r1 = min(max(b, r0), M);
  };
  block_tile_plan<1024>(range, E, max_tiles, max_rows, t, max_small, sh);
}

hipError_t launch_tile_map(const int* offs, int E, int M, int max_rows, void* ws, bool with_small,
                           hipStream_t stream) {
  return launch_k(false, tile_map_kernel, dim3(1), dim3(1024), 0, stream, offs, E, M, max_row_tiles(M, E),
                  max_rows, tile_table_in(ws, M, E), with_small ? max_small_tiles(M, E) : 0);
}

// ---------------------------------------------------------------------------
// Launchers.
// ---------------------------------------------------------------------------
int gemm_max_qtiles(int M, int E) { return max_row_tiles(M, E); }

int gemm_fwd_tile_rows() { return kFwdTileRows; }

static size_t al256(size_t b) { return (b + 255) & ~(size_t)255; }

// The tile plan: header, split-tile counters, tile table, small-tile table.
// Never smaller for more rows or experts.
size_t gemm_plan_bytes(int64_t M, int E) {
  return sizeof(int4) + kSplitTiles * sizeof(int) +
         (size_t)(max_row_tiles((int)M, E) + small_table_tiles(M, E)) * sizeof(int4) + 256;
}

// Partial sums of the split leftover tiles: one piece per workgroup at most.
static size_t gemm_split_bytes() { return (size_t)((num_cus() + 7) & ~7) * kSplitPartBytes; }

// GEMM workspace: the tile plan, then the partial-sum area.
size_t gemm_workspace_bytes(int64_t M, int E) { return al256(gemm_plan_bytes(M, E)) + gemm_split_bytes(); }

static float* split_part_in(void* ws, int M, int E) { return (float*)((char*)ws + al256(gemm_plan_bytes(M, E))); }

// One probe per host thread: a thread's arming stamps only the launches
// that thread makes (other threads' launches never see it).
Probe& probe() {
  thread_local Probe p;
  return p;
}

void gemm_probe_arm(hipEvent_t start, hipEvent_t end) {
  probe().gemm_start = start;
  probe().gemm_end = end;
}

void probe_chain_arm(const hipEvent_t* events, int n_launches) {
  Probe& p = probe();
  p.chain_n = p.chain_i = 0;
  for (int i = 0; i < 2 * n_launches; ++i) p.chain[i] = events[i];
  p.chain_n = n_launches > 0 ? n_launches : 0;
}

// Token tiles of at most h rows that M rows over E experts make, near-even
// loads: every hit expert's share of the rows in whole tiles, or, with fewer
// rows than a tile each, the row count with a partial tile for every third.
static int64_t expected_qtiles(int M, int E, int h) {
  const int64_t hit = std::max(1, std::min(E, M));
  return std::max<int64_t>(hit * ((M + h * hit - 1) / (h * hit)), (M + h - 1) / h + (hit - 1) / 3);
}
static int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Weight rows per tile if a bf16 forward GEMM over `cols` weight rows of k
// columns per expert takes the small-tile kernel, 0 if the large one (320 x
// 256).
//
// Up to kSmallAvgRows rows per expert on average the GEMM streams weights.
// Measured on w13 / w2, us, small against large: 128 experts of 768 x 2048
// with an even load, 2 rows each 127 / 66 against 129 / 69, 40 rows 152 / 89
// against 147 / 88, 100 rows 171 / 104 against 160 / 103; with a Zipf(0.8)
// load 72 rows 173 / 100 against 218 / 103; 32 experts of 7168 x 2048, 9 rows
// 306 / 166 against 307 / 179, 88 rows 324 / 195 against 326 / 195, Zipf(1.2)
// 72 rows 381 / 199 against 319 / 194.  So an even load is about a tie, the
// small tiles are ahead where few long segments leave the large ones ragged,
// and behind where their own tiles just pass a round; the load is not known
// here, and they stay.  At 128 rows many experts need a second 128-row tile
// (even 207 / 117 against 164 / 108) and the large ones are taken.
//
// With more rows per expert the small tiles pay where the large ones leave
// the chip idle in their last round and the weights are re-read from the
// memory-side cache (256 MB): the rounds of each tiling are weighed with its
// time per 64-k stage (0.01 us, 320 x 256: 200, 128 x 256: 108, 128 x 128: 66,
// 64 x 256: 85, 64 x 128: 50); weights that stream from HBM or two and more
// rounds of large tiles are left alone.
//
// In both cases the large tiles may be ahead all the same: by their tail
// split (a reduction cut over workgroups that would idle) and where their
// tiles have less than 320 rows.  Both sides are therefore estimated in time
// (fixed cost per tile, time per stage, the weights' stream; for the split
// its share of the stages and the partial sums), with constants from runs of
// 1 to 4 experts of 5120 x 8192, 16384 x 5120, 7168 x 2048, 2048 x 4096, 2048
// x 768 and 1536 x 2048 with 8 to 8192 rows, and the small ones dropped where
// they lose by 7 %.  One expert, large against small: 5120 x 8192, 8 rows 33
// against 44 us, 64 rows 38 against 53, 800 rows 94 against 109, 4000 rows
// 272 against 368; 16384 x 5120, 320 rows 86 against 100; small ahead: 5120 x
// 8192, 320 rows 59 against 91, 16384 x 5120, 64 rows 37 against 43, 1536 x
// 2048, 500 rows 17 against 48.
constexpr int64_t kSmallWeightBytes = 256 << 20;
static int small_tile_cols(int M, int E, int64_t cols, int k) {
  const int rows = small_tile_rows(M, E);
  if (rows == 0) return 0;
  const int64_t G = (num_cus() + 7) & ~7, stages = k / 64;
  const int64_t large_q = expected_qtiles(M, E, kFwdTileRows), large_tiles = large_q * ceil_div(cols, 256);
  const int64_t weights = std::min(E, M) * cols * k * 2;
  auto rounds = [&](int c) { return ceil_div(expected_qtiles(M, E, rows) * ceil_div(cols, c), G); };
  const int64_t c128 = rounds(128) * (rows == 64 ? 50 : 66), c256 = rounds(256) * (rows == 64 ? 85 : 108);
  const int small = c128 < c256 ? 128 : 256;
  const bool few_rows = M <= kSmallAvgRows * (int64_t)E;
  if (few_rows && large_tiles >= G) return small;
  if (!few_rows && (weights > kSmallWeightBytes || large_tiles >= 2 * G ||
                    std::min(c128, c256) >= ceil_div(large_tiles, G) * 200))
    return 0;
  // 0.01 us
  const int64_t stream = weights / (weights > kSmallWeightBytes ? 60000 : 130000);
  const int64_t small_time = std::min(rounds(128) * (rows == 64 ? 160 + (M <= 32 * (int64_t)E ? 29 : 37) * stages : 230 + 55 * stages),
                                      rounds(256) * (rows == 64 ? 160 + 60 * stages
                                                                : 450 + (rounds(256) > 1 ? 93 : 83) * stages));
  const int64_t h = std::min<int64_t>(kFwdTileRows, (ceil_div(M, large_q) + 31) & ~31);
  const int64_t fixed = 100 + 23 * h / 10, work = stages * std::max<int64_t>(107, 150 * h / 256);
  const int64_t R = large_tiles / G, rt = large_tiles - R * G;
  const int np = split_pieces((int)R, (int)rt, (int)G, (int)stages, split_max());
  // partial sums of a split: cheaper with few leftover tiles
  const int64_t partials = h * (50 + 12 * np) * std::min<int64_t>(std::max<int64_t>(rt, 6), 20) / 200 + 300;
  const int64_t large_time = np > 1 ? R * (fixed + work) + fixed + work / np + partials : (R + (rt > 0)) * (fixed + work);
  return 100 * (600 + std::max(small_time, stream)) > 107 * (600 + std::max(large_time, stream * 105 / 100)) ? 0 : small;
}

// The fp8 tiling: 64-row small tiles (rows 64) or large ones (256) where the
// rows alone decide it, else 128-row small tiles or large ones by the plan's
// tile counts (rows 128: fp8_pick_small, on the device).  Times as in
// small_tile_cols, of the fp8 kernels: 0.01 us per stage of 128 k and tile of
// full height 64 x 128 50, 64 x 256 83, 128 x 128 77, 128 x 256 110, 256 x 256
// 164 and at least 97; with weights that stream from HBM, where a stage waits
// for its rows, 60, 100, 100, 160 and at least 163 (32 experts of 4096 x 7168,
// full rounds; the wider small tile then).  From 1 and 4 experts of 7168 x 2048, 4096 x 7168, 2048 x 1024
// and 2048 x 4096 with 8 to 8000 rows.  Small against large, us: 4 experts of
// 2048 x 4096, 2000 rows 49 against 67, 5000 rows 89 against 69, 8000 rows 95
// against 67; one of 4096 x 7168, 1000 rows 57 against 110, 3000 rows 148
// against 111.
struct Fp8Choice {
  int rows, cols, small_time;
  bool stream;
};
static Fp8Choice fp8_choice(int M, int E, int64_t cols, int k) {
  const int rows = small_tile_rows(M, E), stages = k / 128;
  const bool stream = std::min(E, M) * cols * k > kSmallWeightBytes;
  if (rows == 0) return {kFp8TileRows, 256, 0, stream};
  const int64_t G = (num_cus() + 7) & ~7;
  auto rounds = [&](int c) { return ceil_div(expected_qtiles(M, E, rows) * ceil_div(cols, c), G); };
  if (rows == 64) {
    const int64_t c128 = rounds(128) * (450 + (stream ? 60 : 50) * stages);
    const int64_t c256 = rounds(256) * (493 + (stream ? 100 : 83) * stages);
    const int64_t large_q = expected_qtiles(M, E, kFp8TileRows), large_tiles = large_q * ceil_div(cols, 256);
    const int64_t large = ceil_div(large_tiles, G) * fp8_large_round(stages, stream, (int)ceil_div(M, large_q));
    if (large_tiles < G && 100 * std::min(c128, c256) > 107 * large) return {kFp8TileRows, 256, 0, stream};
    return {64, c128 < c256 ? 128 : 256, 0, stream};
  }
  const int t128 = 50 + 65 * stages, t256 = 100 + (stream ? 137 : 86) * stages;
  const int h = (int)ceil_div(M, expected_qtiles(M, E, 128));
  const bool narrow = !stream && rounds(128) * (t128 + fp8_small_rows(stages, 128, h)) <
                                     rounds(256) * (t256 + fp8_small_rows(stages, 256, h));
  return narrow ? Fp8Choice{128, 128, t128, false} : Fp8Choice{128, 256, t256, stream};
}

// The tiles a forward GEMM with these host counts runs on (ttamd_gemm_tiles).
void gemm_tiles(const int* counts, int E, int64_t weight_rows, int k, bool fp8, int* tile_rows, int* tile_cols,
                int* pieces) {
  int64_t M = 0;
  for (int e = 0; e < E; ++e) M += counts[e];
  *pieces = 1;
  const int G = (num_cus() + 7) & ~7;
  auto tiles_in = [&](int max_rows) {
    int n = 0;
    for (int e = 0; e < E; ++e) n += tiles_of(counts[e], max_rows);
    return n;
  };
  if (fp8) {
    const Fp8Choice c = fp8_choice((int)M, E, weight_rows, k);
    const Fp8Pick p = {nullptr, nullptr, (int)ceil_div(weight_rows, c.cols), c.cols, c.small_time, (int)M, c.stream};
    const bool small = c.rows == 64 || (c.rows == 128 && fp8_pick_small(p, tiles_in(128), tiles_in(kFp8TileRows),
                                                                        (int)ceil_div(weight_rows, 256), k / 128, G));
    *tile_rows = small ? c.rows : kFp8TileRows;
    *tile_cols = small ? c.cols : 256;
    return;
  }
  const int small = small_tile_cols((int)M, E, weight_rows, k);
  *tile_rows = small ? small_tile_rows((int)M, E) : kFwdTileRows;
  *tile_cols = small ? small : 256;
  if (small) return;
  const int64_t tiles = tiles_in(kFwdTileRows) * ceil_div(weight_rows, 256);
  if (tiles / G <= kSplitMaxRounds) *pieces = split_pieces((int)(tiles / G), (int)(tiles % G), G, k / 64, split_max());
}

// plan: the tile plan; part: the partial-sum area of split leftover tiles
// (nullable: no split).  table_ready: `plan` already holds the tile table
// of these rows (built for kFwdTileRows-row tiles), so no tile-map launch.
static hipError_t fwd(int epi, FwdGemm g, const int* offs, int E, int M, void* plan, float* part,
                      hipStream_t stream, bool table_ready = false) {
  if (!table_ready) {
    hipError_t err = launch_tile_map(offs, E, M, kFwdTileRows, plan, true, stream);
    if (err != hipSuccess) return err;
  }
  const TileTable tt = tile_table_in(plan, M, E);
  const int small = small_tile_cols(M, E, epi == EPI_SWIGLU ? 2 * (int64_t)g.n : g.n, g.kred);
  g.table = small ? tt.small_table : tt.table;
  g.n_qtiles = small ? tt.small_count : tt.count;
  g.split_cnt = tt.split_cnt;
  g.part = part;
  return launch_fwd_gemm(epi, g, tt.small_rows, small, stream);
}
static hipError_t fwd(int epi, FwdGemm g, const int* offs, int E, int M, void* ws, hipStream_t stream) {
  return fwd(epi, g, offs, E, M, ws, split_part_in(ws, M, E), stream);
}

hipError_t launch_grouped_mm(const void* x, const void* w, const int* offs, int M, int E,
                             int N, int K, void* out, void* ws, hipStream_t stream) {
  FwdGemm g = {};
  g.act = x; g.w = w; g.kred = K; g.n = N; g.out = out;
  return fwd(EPI_STORE, g, offs, E, M, ws, stream);
}

hipError_t launch_grouped_mm_swiglu(const void* x, const void* w13, const int* offs, int M,
                                    int E, int H, int D, float limit, void* a_out, void* h_out,
                                    void* ws, hipStream_t stream) {
  FwdGemm g = {};
  g.act = x; g.w = w13; g.kred = D; g.n = H; g.out = a_out; g.limit = limit; g.h_out = h_out;
  return fwd(EPI_SWIGLU, g, offs, E, M, ws, stream);
}

hipError_t launch_grouped_mm_swiglu_gather(const void* tokens, int n_tokens, const int* src_index,
                                           int src_div, const void* w13, const int* offs, int M, int E,
                                           int H, int D, float limit, void* a_out, void* h_out, void* ws,
                                           hipStream_t stream) {
  FwdGemm g = {};
  g.act = tokens; g.act_index = src_index; g.act_div = src_div; g.n_act = n_tokens;
  g.w = w13; g.kred = D; g.n = H; g.out = a_out; g.limit = limit; g.h_out = h_out;
  return fwd(EPI_SWIGLU, g, offs, E, M, ws, stream);
}

hipError_t launch_grouped_mm_unpermute(const void* act, const void* w2, const int* offs, int M,
                                       int E, int D, int H, const float* row_scale,
                                       const int* dest, int n_dest, void* out, void* ws,
                                       hipStream_t stream) {
  FwdGemm g = {};
  g.act = act; g.w = w2; g.kred = H; g.n = D; g.out = out;
  g.row_scale = row_scale; g.dest = dest; g.n_dest = n_dest;
  return fwd(EPI_SCATTER, g, offs, E, M, ws, stream);
}

// ---- the expert stage of the MoE layer forward in one call ---------------------
size_t moe_experts_forward_workspace_bytes(int64_t T, int64_t D, int64_t H, int E, int K, bool permute_first) {
  const int64_t M = T * K;
  auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
  size_t n = al(gemm_workspace_bytes(M, E));                 // tile plan
  n += al((size_t)M * H * 2);                                // a = swiglu(x w13^T)
  if (permute_first) n += al((size_t)M * D * 2);             // routed rows
  if (K > 1) n += al((size_t)M * D * 2);                     // y in flat-slot order
  return n;
}

hipError_t launch_moe_experts_forward(const void* tokens, int T, int D, int H, int E, int K,
                                      const int* sorted_idx, const int* offs, const float* sorted_scores,
                                      bool score_before, float limit, const void* w13, const void* w2,
                                      void* out, void* plan, void* ws, hipStream_t stream) {
  const int M = T * K;
  const bool permute_first = score_before || D < 128;
  auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
  char* p = (char*)ws;
  void* own_plan = p;
  p += al(gemm_workspace_bytes(M, E));
  void* a = p;
  p += al((size_t)M * H * 2);
  void* routed = nullptr;
  if (permute_first) {
    routed = p;
    p += al((size_t)M * D * 2);
  }
  void* y = (K > 1) ? (void*)p : out;
  hipError_t err;
  // one tile table for both GEMMs
  void* tp = plan;
  float* part = split_part_in(own_plan, M, E);
  if (tp == nullptr) {
    tp = own_plan;
    if ((err = launch_tile_map(offs, E, M, kFwdTileRows, tp, true, stream)) != hipSuccess) return err;
  }
  if (permute_first) {
    err = launch_gather_rows(tokens, sorted_idx, score_before ? sorted_scores : nullptr, false, T, M, M, D, K,
                             routed, stream);
    if (err != hipSuccess) return err;
    FwdGemm g = {};
    g.act = routed; g.w = w13; g.kred = D; g.n = H; g.out = a; g.limit = limit;
    err = fwd(EPI_SWIGLU, g, offs, E, M, tp, part, stream, true);
  } else {
    FwdGemm g = {};
    g.act = tokens; g.act_index = sorted_idx; g.act_div = K; g.n_act = T;
    g.w = w13; g.kred = D; g.n = H; g.out = a; g.limit = limit;
    err = fwd(EPI_SWIGLU, g, offs, E, M, tp, part, stream, true);
  }
  if (err != hipSuccess) return err;
  FwdGemm g2 = {};
  g2.act = a; g2.w = w2; g2.kred = H; g2.n = D; g2.out = y;
  g2.row_scale = score_before ? nullptr : sorted_scores;
  g2.dest = sorted_idx;
  g2.n_dest = (K > 1) ? M : T;
  if ((err = fwd(EPI_SCATTER, g2, offs, E, M, tp, part, stream, true)) != hipSuccess) return err;
  if (K > 1) return launch_combine(y, nullptr, nullptr, T, K, D, out, stream);
  return hipSuccess;
}

// ---- fp8 forward (gemm_fp8.hip) ----------------------------------------------
static hipError_t fp8(int epi, Fp8Args a, const int* offs, int E, int M, void* ws,
                      hipStream_t stream) {
  hipError_t err = launch_tile_map(offs, E, M, kFp8TileRows, ws, true, stream);
  if (err != hipSuccess) return err;
  const TileTable tt = tile_table_in(ws, M, E);
  const Fp8Choice c = fp8_choice(M, E, a.n_p, a.kred);
  a.table = c.rows == 64 ? tt.small_table : tt.table;
  a.n_qtiles = c.rows == 64 ? tt.small_count : tt.count;
  const Fp8Pick p = {tt.small_table, tt.small_count, 0, c.cols, c.small_time, M, c.stream};
  return launch_fp8_gemm(epi, a, p, c.rows, c.cols, stream);
}

static Fp8Args fp8_args(const void* xq, const float* sx, const void* wq, const float* sw, int M,
                        int N_rows, int K) {
  Fp8Args a = {};
  a.q = (const uint8_t*)xq;
  a.ldq = K;
  a.p = (const uint8_t*)wq;
  a.p_estride = (int64_t)N_rows * K;
  a.ldp = K;
  a.kred = K;
  a.sx = sx;
  a.ldsx = M;
  a.sw = sw;
  a.sw_estride = (int64_t)(N_rows / 128) * (K / 128);
  return a;
}

hipError_t launch_grouped_mm_fp8(const void* xq, const float* sx, const void* wq, const float* sw,
                                 const int* offs, int M, int E, int N, int K, void* out, void* ws,
                                 hipStream_t stream) {
  Fp8Args a = fp8_args(xq, sx, wq, sw, M, N, K);
  a.np_tiles = (N + 255) / 256;
  a.n_p = N;
  a.out = (bf16_t*)out;
  a.ldo = N;
  return fp8(EPI_STORE, a, offs, E, M, ws, stream);
}

hipError_t launch_grouped_mm_fp8_swiglu(const void* xq, const float* sx, const void* w13q,
                                        const float* s13, const int* offs, int M, int E, int H, int D,
                                        float limit, void* a_out, void* h_out, void* ws,
                                        hipStream_t stream) {
  Fp8Args a = fp8_args(xq, sx, w13q, s13, M, 2 * H, D);
  a.np_tiles = (H + 127) / 128;  // 128 gate + 128 up rows per tile (H % 64 == 0)
  a.n_p = 2 * H;
  a.out = (bf16_t*)a_out;
  a.ldo = H;
  a.hidden = H;
  a.limit = limit;
  a.h_out = (bf16_t*)h_out;
  a.ldh = 2 * (int64_t)H;
  return fp8(EPI_SWIGLU, a, offs, E, M, ws, stream);
}

hipError_t launch_grouped_mm_fp8_unpermute(const void* aq, const float* sa, const void* w2q,
                                           const float* s2, const int* offs, int M, int E, int D, int H,
                                           const float* row_scale, const int* dest, int n_dest,
                                           void* out, void* ws, hipStream_t stream) {
  Fp8Args a = fp8_args(aq, sa, w2q, s2, M, D, H);
  a.np_tiles = (D + 255) / 256;
  a.n_p = D;
  a.out = (bf16_t*)out;
  a.ldo = D;
  a.row_scale = row_scale;
  a.dest = dest;
  a.n_dest = n_dest;
  return fp8(EPI_SCATTER, a, offs, E, M, ws, stream);
}

static hipError_t dgrad(int epi, DgradGemm g, const int* offs, int E, int M, void* plan, float* part,
                        hipStream_t stream) {
  hipError_t err = launch_tile_map(offs, E, M, kFwdTileRows, plan, false, stream);
  if (err != hipSuccess) return err;
  const TileTable tt = tile_table_in(plan, M, E);
  g.table = tt.table;
  g.n_qtiles = tt.count;
  g.split_cnt = tt.split_cnt;
  g.part = part;
  return launch_dgrad_gemm(epi, g, stream);
}

hipError_t launch_shared_expert_add(const void* x, int T, int D, int H, const void* w13s, const void* w2s,
                                   const float* gate_logits, float limit, void* a_scratch, void* out,
                                   void* ws, hipStream_t stream) {
  // one expert with all T rows: a = swiglu(x w13s^T), then out += g(t) * (a w2s^T)
  FwdGemm g1 = {};
  g1.act = x; g1.w = w13s; g1.kred = D; g1.n = H; g1.out = a_scratch; g1.limit = limit;
  hipError_t err = fwd(EPI_SWIGLU, g1, nullptr, 1, T, ws, stream);
  if (err != hipSuccess) return err;
  FwdGemm g2 = {};
  g2.act = a_scratch; g2.w = w2s; g2.kred = H; g2.n = D; g2.out = out; g2.n_dest = T;
  g2.row_scale = gate_logits; g2.scale_sigmoid = 1; g2.accumulate = 1;
  return fwd(EPI_SCATTER, g2, nullptr, 1, T, ws, stream);
}

hipError_t launch_grouped_mm_dgrad(const void* dy, const void* w, const int* offs, int M, int E,
                                   int N, int K, void* dx, void* ws, hipStream_t stream) {
  // dx[m][k] = sum_n dy[m][n] w[e][n][k]
  DgradGemm g = {};
  g.dy = dy; g.w = w; g.n_red = N; g.n_out = K; g.out = dx;
  return dgrad(EPI_STORE, g, offs, E, M, ws, split_part_in(ws, M, E), stream);
}

hipError_t launch_grouped_mm_dgrad_unsplit(const void* dy, const void* w, const int* offs, int M, int E, int N,
                                           int K, void* dx, void* plan, hipStream_t stream) {
  DgradGemm g = {};
  g.dy = dy; g.w = w; g.n_red = N; g.n_out = K; g.out = dx;
  return dgrad(EPI_STORE, g, offs, E, M, plan, nullptr, stream);
}

hipError_t launch_grouped_mm_dgrad_swiglu(const void* dy, const void* w2, const void* h,
                                          const int* offs, int M, int E, int D, int H,
                                          float limit, void* dh, void* a_out, void* ws,
                                          hipStream_t stream) {
  // g[m][p] = sum_d dy[m][d] w2[e][d][p], then the SwiGLU backward with h
  DgradGemm g = {};
  g.dy = dy; g.w = w2; g.n_red = D; g.n_out = H; g.out = dh; g.h = h; g.limit = limit; g.a_out = a_out;
  return dgrad(EPI_SWIGLU_BWD, g, offs, E, M, ws, split_part_in(ws, M, E), stream);
}

hipError_t launch_grouped_mm_wgrad(const void* dy, const void* x, const int* offs, int M, int E,
                                   int N, int K, void* dw, bool fp32, void* ws, hipStream_t stream) {
  WgradDmaArgs a = {};
  a.dy = (const bf16_t*)dy; a.lddy = N;
  a.x = (const bf16_t*)x; a.ldx = K;
  a.offs = offs; a.E = E; a.M = M; a.N = N; a.K = K;
  a.n_tiles = (N + 255) / 256; a.k_tiles = (K + 255) / 256;
  a.dw = dw; a.dw_fp32 = fp32 ? 1 : 0;
  a.split_np = 1;
  if (ws != nullptr) {
    // Tail split for a walk of at most kSplitMaxRounds full rounds with
    // tiles left over: up to kSplitMaxPieces pieces per leftover tile, so
    // that the pieces fill the otherwise idle workgroups, each piece of at
    // least kSplitMinStages stages of the average expert's rows.
    const int G = (num_cus() + 7) & ~7;
    const int ntiles = E * a.n_tiles * a.k_tiles;
    const int R = ntiles / G, rt = ntiles - R * G;
    if (rt > 0 && rt <= kSplitTiles && R <= kSplitMaxRounds) {
      int np = std::min(kSplitMaxPieces, G / rt);
      const int avg_stages = (M / E + 63) / 64;
      while (np > 1 && avg_stages < np * kSplitMinStages) --np;
      if (np > 1) {
        TileTable tt = tile_table_in(ws, M, E);
        hipError_t err = launch_split_cnt_zero(tt.split_cnt, rt, stream);
        if (err != hipSuccess) return err;
        a.part = split_part_in(ws, M, E);
        a.split_cnt = tt.split_cnt;
        a.split_np = np;
      }
    }
  }
  return launch_wgrad_dma(a, stream);
}

}  // namespace ttamd
