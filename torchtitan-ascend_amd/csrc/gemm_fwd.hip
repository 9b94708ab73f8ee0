// Persistent grouped GEMM for the expert FFN forward on MI355X (gfx950).
//
//   out[q, p] = sum_k act[q, k] * w[e(q), p, k]        (k contiguous in both)
//
// q runs over routed token rows grouped by expert (ragged segments), p over
// weight rows.  Used for the w13 up-projection with SwiGLU fused into the
// epilogue, for the w2 down-projection with the routing-weight scale and the
// un-permute scatter fused into the epilogue, and for the plain grouped GEMM.
//
// Tile: up to 320 token rows (Q) x 256 weight rows (P); k in stages of 64.
//   * 8 waves, two per SIMD, in a 2 x 4 arrangement: wave (wq, wp) owns 64
//     weight rows and 16 rows of each of the tile's 32-row token blocks (up
//     to 10; 4 x 10 accumulators of v_mfma_f32_16x16x32_bf16, 160 fp32
//     registers per lane).  The block count follows the tile's height (the
//     k loop is instantiated per count), so a 256-row tile costs 256 rows of
//     MFMA, LDS reads and token-row DMA, not 320.  The MFMA A operand is the
//     weight tile, B the token tile, so a lane holds 4 consecutive output
//     columns per block.  SWIGLU: a wave's weight rows are 32 gate rows and
//     the 32 matching up rows.
//   * Two LDS stage buffers of 72 KB (32 KB weights + 40 KB tokens, rows of
//     128 bytes = one full cache line per row and stage) filled by
//     global_load_lds_dwordx4 (HBM/L2 -> LDS without VGPR staging).  A DMA
//     instruction moves 8 whole rows; half-line rows (k stages of 32) cost
//     twice the L2 requests per byte and capped the load rate.  The 16-byte
//     chunk c of row r sits at c ^ ((r ^ (r >> 3)) & 7), which keeps the
//     fragment reads free of bank conflicts.  A wave's DMA writes 1 KB of LDS
//     contiguously, so the permutation is applied to the global addresses.
//   * A stage is worked off token block by token block, with all of its
//     weight fragments in registers.  Its weight rows and first token blocks
//     are therefore free early, and the next-but-one stage's DMAs into them
//     are in flight for almost two stages; they go out one at a time between
//     the MFMAs (run_tile).
//   * What bounds it: at C3 w13 the chip runs at 1.96 GHz (it lowers its
//     clock under MFMA load) with the matrix cores 64 % busy over the launch
//     (w2 59 %; C2, whose tiles have 32 and 12 stages, 54 and 42 %), the rest
//     lost around a stage's two barriers, in the epilogues and in the last
//     round.  Measured, one machine, against 32x32x16 MFMAs
//     over k16 steps with each stage's DMAs issued in two bursts: C2 w13 401
//     -> 381 us, w2 245 -> 235, dgrad + SwiGLU backward 344 -> 279; C3 w13
//     1257 -> 1183, w2 676 -> 633, dgrad + SwiGLU backward 768 -> 699, dgrad
//     1326 -> 1267; C4 w13 1642 -> 1549, w2 904 -> 850 us.
//   * Per tile, a wave-uniform byte base (SGPRs) plus one 32-bit per-lane
//     offset per DMA instruction; per stage only the k offset changes.
//   * Persistent: one workgroup per CU walks the tile list with stride
//     gridDim.x; the DMA stream runs over the flattened (tile, k-stage)
//     sequence, so the next tile's first stages load during the current
//     tile's epilogue.  Within a round the 32 workgroups of one XCD take 32
//     consecutive tiles (same expert), so the weights are shared in its L2
//     (the SwiGLU kernels walk the token tiles in pairs, see tile_at).
//   * Tail split: for a walk of at most six full rounds, the tiles left
//     over after the last full round are cut along k into up to 8 pieces
//     that run on the otherwise idle workgroups; every piece writes its fp32
//     accumulators to the workspace and counts its arrival (agent-scope
//     release / atomic / acquire, as the XCDs' L2s are not coherent), and
//     the last piece to arrive streams all partials back through LDS in
//     piece order, so the sum does not depend on arrival order, and runs the
//     ordinary epilogue.
//
// Reference semantics (torchtitanturbo/models/common/npu_gmm.py):
//   :17-18, :31, :38  torch._grouped_mm(x, w.transpose(-2, -1), offs)
//   :32-36            optional clamp with swiglu_limit
//   :37               npu_swiglu: silu(gate) * up, gate = first H columns
#include <cstddef>
#include <cstdlib>
#include <type_traits>

#include "common.h"
#include "dma_asm.h"
#include "gemm_common.h"
#include "kernels.h"

namespace ttamd {
namespace {

using namespace dma;

constexpr int TQ = kFwdTileRows;  // 320 token rows
constexpr int TP = 256;           // weight rows
constexpr int WAVES = 8;          // 2 per SIMD
constexpr int WPN = WAVES / 2;    // waves along the weight rows (2 along the token rows)
constexpr int NJ = TQ / 32;       // 16-row token blocks per wave
constexpr int NPB = TP / 16 / WPN;  // 16-row weight blocks per wave
constexpr int TK = 64;            // k per stage: 128-byte rows
constexpr int NSTAGE = 2;
constexpr int FTHREADS = 64 * WAVES;
constexpr int ROW_BYTES = TK * 2;
constexpr int P_BYTES = TP * ROW_BYTES;                // 32 KB
constexpr int STAGE_BYTES = P_BYTES + TQ * ROW_BYTES;  // 72 KB
constexpr int LDS_BYTES = NSTAGE * STAGE_BYTES;        // 144 KB
constexpr int DMA_P = TP / 8 / WAVES;                  // 4 weight-row instructions per wave
constexpr int DMA_Q = TQ / 8 / WAVES;                  // 5 token-row instructions per wave
constexpr int QA = 2;  // token-row instructions issued with a stage's weight rows
static_assert(TQ % 64 == 0 && TP == 256 && TQ % (8 * WAVES) == 0 && NPB == 4, "tile geometry");
// EPI_SCATTER row metadata (destination row, scale) of a tile, DMA'd with
// the tile's first stage into one of three LDS slots (tile round % 3): the
// slot of round r + 3 is written only after round r's epilogue.
constexpr int META_BYTES = TQ * 8;
// Gathered token rows (q_index): the tile's source-row ids, DMA'd one tile
// ahead into one of two LDS slots (tile round % 2), and the byte offsets of
// the rows being issued, which every wave keeps for the rows it moves.
constexpr int IDX_OFF = LDS_BYTES + 3 * META_BYTES;
constexpr int IDX_BYTES = TQ * 4;
constexpr int GOFF_OFF = IDX_OFF + 2 * IDX_BYTES;
constexpr int LDS_TOTAL = GOFF_OFF + IDX_BYTES;  // 155 KB
// Split tail tiles: whether this workgroup's piece arrived last, in the
// stage buffers (free by then) past the ring the partial sums stream through.
constexpr int FLAG_OFF = 8 * 16 * 1024;
static_assert(FLAG_OFF + 16 <= LDS_BYTES, "flag inside the stage buffers");
static_assert(kSplitPartBytes == (size_t)WAVES * NJ * NPB * 4 * 64 * 4, "partial-sum area of a piece");

typedef short short4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) short4_t lds_short4_t;
typedef __attribute__((address_space(1))) int gint_t;
typedef __attribute__((address_space(1))) floatx4_t gfloatx4_t;

// Chunk permutation of the 512-byte reduction-major weight rows (PT): the 16
// rows 16 g + 8 t + 4 h .. + 3 (g = 0..3) that one transposed read touches, 32
// bytes each, land on eight distinct 32-byte bank groups, two rows each.
__device__ __forceinline__ int ptswz(int n) { return 2 * ((n & 3) | ((n >> 2) & 4)); }

// f(integral_constant) for A, A + 1, ..., B - 1.
template <int A, int B, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (A < B) {
    f(std::integral_constant<int, A>{});
    static_for<A + 1, B>(f);
  }
}

// PT (dgrad): the weight operand is reduction-major, w[e][n][k] with the
// reduction n as rows and the output index k contiguous.  Its stage is 64
// rows of TP * 2 = 512 bytes (n rows of the tile's 256 output columns), the
// 16-byte chunk c of row n stored at c ^ ptswz(n), and the MFMA A fragments
// (8 consecutive n for one output column) come from two
// ds_read_b64_tr_b16 per block: within each 16-lane group, lane i receives
// element i % 4 of the 4 loaded by lane 4c + i / 4, for c = 0..3, so lane
// src points at row n0 + src / 4, columns r0 + 4 (src % 4) .. + 3, and lane
// i receives rows n0 .. n0 + 3 of column r0 + i.
// GATHER (inference w13): token row j is q row q_index[j] / q_div.
template <int EPI, bool PT, bool GATHER>
__global__ __launch_bounds__(FTHREADS, 1) void gg_fwd_kernel(const FwdArgs a) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wq = w / WPN;
  const int wp = w % WPN;
  const int l = threadIdx.x & 63;
  const int G = gridDim.x;
  const int b = blockIdx.x;
  // XCD-aware slot: hardware block ids go round-robin over the 8 XCDs; give
  // XCD x the slots [x*G/8, (x+1)*G/8) so that it takes consecutive tiles.
  const int slot = (b & 7) * (G >> 3) + (b >> 3);
  const int nqt = sload_int(a.n_qtiles);
  const int ntiles = nqt * a.np_tiles;
  // (the schedule scalars are pinned to SGPRs: divisions are expanded in
  // VALU, and issue_advance must stay scalar)
  auto U = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
  const int ksteps = U(a.kred / TK);
  // Tail split: the walk has R full rounds of G tiles and rt tiles left
  // over.  Unsplit, rt workgroups run one more whole tile while the others
  // idle.  Split, each leftover tile is cut along k into np pieces of
  // consecutive stages, piece j of leftover tile t taken by slot j * rt + t
  // (so one XCD's slots run the same k range of neighbouring tiles), and
  // every slot runs R whole tiles, then at most one piece.
  const int R = U(ntiles / G);
  const int rt = ntiles - R * G;
  const int np = a.part != nullptr ? U(split_pieces(R, rt, G, ksteps, a.split_max)) : 1;
  const bool has_piece = np > 1 && slot < rt * np;
  const int nfull = U(np > 1 ? R : (slot < ntiles ? (ntiles - slot + G - 1) / G : 0));
  const int nmy = nfull + (has_piece ? 1 : 0);
  const int pc_t = has_piece ? slot % rt : 0;  // leftover tile of the piece
  const int pc_j = has_piece ? slot / rt : 0;  // piece index
  const int pc_k0 = U(pc_j * ksteps / np);
  const int pc_k1 = U((pc_j + 1) * ksteps / np);
  const int pc_L = U(R * G + pc_t);  // its walk index
  // np, pc_j and pc_t in one register through the k loop (unpacked after it)
  const int pc_info = U(np | (pc_j << 8) | (pc_t << 16));
  // Persistent order of the SwiGLU (w13) kernels: token tiles in pairs,
  // weight tile major inside a pair, so 32 consecutive slots (one XCD's)
  // take both token tiles of an expert with 16 weight tiles rather than one
  // token tile with 32: each weight tile is shared in the XCD's L2 instead
  // of across XCDs (C3 w13 -6 %; the other epilogues' kernels were slower
  // with it and keep the table order).  Returns the table order's tile id
  // (qt * np_tiles + pt).
  auto tile_at = [&](int r) {
    const int L = r < nfull ? r * G + slot : pc_L;
    if constexpr (EPI != EPI_SWIGLU) return L;
    const int blk = L / (2 * a.np_tiles);
    const int in_blk = L - blk * 2 * a.np_tiles;
    const int gq = min(2, nqt - 2 * blk);
    const int pt = in_blk / gq;
    return (2 * blk + (in_blk - pt * gq)) * a.np_tiles + pt;
  };
  const int total = nfull * ksteps + (has_piece ? pc_k1 - pc_k0 : 0);
  if (total == 0) return;

  const uint32_t lds0 = lds_addr(smem);
  // DMA lane geometry: instruction i of wave w (per operand) writes the 8
  // rows of row block rb = WAVES*i + w, row 8rb + l / 8, physical chunk l % 8,
  // whose logical chunk is l % 8 ^ cswz(row) = l % 8 ^ ((l / 8 ^ rb) & 7).
  const int drow = l >> 3;

  // ---- DMA stream -----------------------------------------------------------
  // Source-row ids of tile round r (gathered rows only): 64-row chunk c of
  // the tile is moved by wave c % WAVES into slot r % 2.
  auto load_ids = [&](int r) {
    const int tile = tile_at(r);
    const int4 ti = sload_int4(a.table + tile / a.np_tiles);
    for (int c = w; c < TQ / 64; c += WAVES) {
      const uint32_t q = (uint32_t)min(64 * c + l, ti.z - ti.y - 1);
      dma4(q * 4, (uint64_t)(a.q_index + ti.y), lds0 + IDX_OFF + (uint32_t)((r & 1) * IDX_BYTES) + c * 256);
    }
  };
  int d_r = -1;  // tile round whose addresses are loaded
  int d_rot = 0;  // its first k stage
  int d_qblk8 = 0;  // 8-row token blocks the MFMA reads: 4 * ceil(rows / 32)
  int d_pmax = 0, d_qmax = 0;  // last valid weight / token row of the tile (tile-relative)
  uint64_t d_pbase = 0, d_qbase = 0;
  // Row-major operands: instruction i of wave w moves rows rr0 + 64 i with
  // the same chunk permutation (row block 8 i + w has (8 i + w) & 7 = w), so
  // its per-lane offset is recomputed at issue from two lane constants and
  // the tile's uniform clamps, instead of occupying a register per
  // instruction through the k loop.  Per-lane offsets that are not affine
  // in i (transposed weights, gathered token rows) are kept per tile.
  static_assert(WAVES == 8, "row block 8 i + w has chunk permutation term w");
  const int rr0 = 8 * w + drow;
  const uint32_t lch16 = (uint32_t)(((l & 7) ^ ((drow ^ w) & 7)) * 16);
  // PT: rows 2 (WAVES i + w) and + 1, 32 chunks each.  The chunk permutation
  // depends on i through bit 3 (i % 2), which is bit 7 of the byte offset
  // (rows are a multiple of 256 bytes apart); otherwise instruction i moves
  // the uniform base.
  uint32_t d_ptoff = 0;
  // GATHER: byte offsets of this wave's rows (instruction i, row l / 8) in LDS
  int* const goff = (int*)(smem + GOFF_OFF) + w * (DMA_Q * 8);
  auto dma_tile = [&](int r) {
    const int tile = tile_at(r);
    const int qt = tile / a.np_tiles;
    const int pt = tile - qt * a.np_tiles;
    const int4 ti = sload_int4(a.table + qt);
    const int64_t ldp2 = a.ldp * 2;
    const int qmax = ti.z - ti.y - 1;
    d_qblk8 = 4 * ((ti.z - ti.y + 31) >> 5);
    d_qmax = qmax;
    if constexpr (PT) {
      const int row = 2 * w + (l >> 5);
      // a tile with 128 valid columns (N % 128 == 0) reads those twice
      const int lc = ((l & 31) ^ ptswz(row)) & (a.n_p - pt * TP >= TP ? 31 : 15);
      d_ptoff = (uint32_t)(row * ldp2 + lc * 16);
    } else {
      d_pmax = a.n_p - 1 - pt * (EPI == EPI_SWIGLU ? 128 : TP);
    }
    if constexpr (GATHER) {
      // Gathered rows: tile row rr reads source row q_index[row] / q_div,
      // whose id was DMA'd into LDS while the previous tile was issued.  Lane
      // 8 i + j works out row j of this wave's instruction i.
      const int* ids = (const int*)(smem + IDX_OFF + (r & 1) * IDX_BYTES);
      if (l < DMA_Q * 8) {
        const int row = min(64 * (l >> 3) + 8 * w + (l & 7), qmax);
        const int src = min(max(ids[row] / a.q_div, 0), a.n_q_in - 1);
        goff[l] = (int)((uint32_t)src * (uint32_t)(a.ldq * 2));
      }
      lds_wait();
      if (r + 1 < nmy) load_ids(r + 1);
    }
    if constexpr (PT)
      d_pbase = (uint64_t)(a.p + (int64_t)ti.x * a.p_estride + (int64_t)pt * TP);
    else if constexpr (EPI == EPI_SWIGLU)
      d_pbase = (uint64_t)(a.p + (int64_t)ti.x * a.p_estride + (int64_t)pt * 128 * a.ldp);
    else
      d_pbase = (uint64_t)(a.p + (int64_t)ti.x * a.p_estride + (int64_t)pt * TP * a.ldp);
    d_qbase = (uint64_t)(a.q + (GATHER ? 0 : (int64_t)ti.y * a.ldq));
    if constexpr (EPI == EPI_SCATTER) {
      for (int c = w; c < TQ / 64; c += WAVES) {
        const uint32_t q = (uint32_t)min(64 * c + l, qmax);
        const uint32_t m = lds0 + LDS_BYTES + (uint32_t)((r % 3) * META_BYTES) + c * 256;
        if (a.dest) dma4(q * 4, (uint64_t)(a.dest + ti.y), m);
        if (a.row_scale) dma4(q * 4, (uint64_t)(a.row_scale + ti.y), m + TQ * 4);
      }
    }
    // Weight rows a multiple of 4 KB apart: tiles at the same k ask the same
    // HBM channels, so each expert starts its k walk elsewhere (the tiles of
    // one expert keep sharing their lines).  Against one k order for all, us:
    // 128 experts of 1536 x 2048, 128 rows each 199 -> 160, 256 rows 228 ->
    // 202, 512 rows 357 -> 353, 1024 rows unchanged; 32 of 7168 x 2048, 128
    // rows 239 -> 200, 512 rows 424 -> 426; 32 of 4096 x 4096, 128 rows 250 ->
    // 198; 16 of 4096 x 6144, 192 rows 203 -> 174.  Not for rows of 16 KB and
    // more, where it loses with few rows per expert and gains nothing with
    // many: 16 of 5120 x 8192, 128 rows 286 -> 299, 512 rows 589 -> 590; 8 of
    // 8192 x 8192, 192 rows 218 -> 242.  Offsets per weight tile as well lose
    // the shared token lines (512 rows 382 -> 407).  A split tile's pieces keep
    // their k ranges.
    if constexpr (!PT) {
      const uint32_t row = (uint32_t)a.ldp * 2;
      d_rot = row % 4096 == 0 && row < 16384 && r < nfull ? U(3 * ti.x % ksteps) : 0;
    }
    d_r = r;
  };
  // A stage's DMAs go out one instruction at a time between the MFMAs of the
  // stage two before it, whose buffer they fill: the weight rows and the first
  // QA token-row instructions after its barrier A, the other token rows after
  // its barrier B (run_tile).  issue_prep sets the bases that issue_p1 and
  // issue_q1 read, issue_advance steps to the next stage.
  uint64_t d_spb = 0, d_sqb = 0;
  uint32_t d_sst = 0;
  // Stages are issued in order, 0, 1, 2, ...: the (unit, k stage) of the next
  // one is advanced rather than divided out per call.  Past the end the last
  // stage is issued again.
  int n_r = 0, n_ks = nfull > 0 ? 0 : pc_k0, n_kend = nfull > 0 ? ksteps : pc_k1, n_left = total;
  auto issue_prep = [&](int s) {
    if (n_r != d_r) dma_tile(n_r);
    int ks = n_ks + d_rot;
    ks = ks >= ksteps ? ks - ksteps : ks;
    d_spb = d_pbase + (PT ? (uint64_t)ks * TK * a.ldp * 2 : (uint64_t)ks * ROW_BYTES);
    d_sqb = d_qbase + (uint64_t)ks * ROW_BYTES;
    d_sst = lds0 + (uint32_t)((s & 1) * STAGE_BYTES) + w * 1024;
  };
  auto issue_p1 = [&](int i) {
    const uint32_t ldp2 = (uint32_t)a.ldp * 2u;
    {
      uint32_t voff;
      if constexpr (PT) {
        dma16(d_ptoff ^ (128u * (i & 1)), d_spb + (uint64_t)(uint32_t)(i * 2 * WAVES) * (uint64_t)(a.ldp * 2), d_sst + i * (WAVES * 1024));
        return;
      } else if constexpr (EPI == EPI_SWIGLU) {
        // rows 0..127 gate, 128..255 up: tile row rr is weight row pt * 128 +
        // (rr & 127), of the up half (hidden + ...) for rr >= 128
        const int col = min(rr0 + 64 * (i & 1), d_pmax);
        voff = (uint32_t)(i < 2 ? col : (int)a.hidden + col) * ldp2 + lch16;
      } else {
        voff = (uint32_t)min(rr0 + 64 * i, d_pmax) * ldp2 + lch16;
      }
      dma16(voff, d_spb, d_sst + i * (WAVES * 1024));
    }
  };
  auto issue_advance = [&]() {
    // Advance to the next stage only after its DMAs: whatever sits between a
    // barrier and the DMAs behind it delays every stage (the empty asm keeps
    // the compiler from hoisting the update above them).  Selects, no branches.
    n_left = __builtin_amdgcn_readfirstlane(n_left);
    n_ks = __builtin_amdgcn_readfirstlane(n_ks);
    n_kend = __builtin_amdgcn_readfirstlane(n_kend);
    n_r = __builtin_amdgcn_readfirstlane(n_r);
    asm volatile("" : "+s"(n_left), "+s"(n_ks), "+s"(n_kend), "+s"(n_r));
    const int adv = n_left > 1 ? 1 : 0;
    n_left -= adv;
    const int nk = n_ks + adv;
    const bool wrap = nk == n_kend;
    n_r += wrap ? 1 : 0;
    const bool full = n_r < nfull;
    n_ks = wrap ? (full ? 0 : pc_k0) : nk;
    n_kend = wrap ? (full ? ksteps : pc_k1) : n_kend;
  };
  // Token rows: instruction i moves the tile's rows 64 i .. + 63.  The first
  // QA always go out (rows past the tile repeat its last row), so the DMAs in
  // flight at a stage barrier can be counted; past the tile's last 32-row
  // block the others are skipped (wave-uniform: instruction i moves row block
  // WAVES * i + w).
  auto issue_q1 = [&](int i) {
    const uint32_t voff = (GATHER ? (uint32_t)goff[8 * i + drow]
                                  : (uint32_t)min(rr0 + 64 * i, d_qmax) * ((uint32_t)a.ldq * 2u)) + lch16;
    const uint32_t dst = d_sst + P_BYTES + i * (WAVES * 1024);
    if (i < QA)
      dma16(voff, d_sqb, dst);
    else if (WAVES * i + w < d_qblk8)
      dma16(voff, d_sqb, dst);
  };
  auto issue_all = [&](int st) {
    issue_prep(st);
#pragma unroll
    for (int i = 0; i < DMA_P; ++i) issue_p1(i);
#pragma unroll
    for (int i = 0; i < DMA_Q; ++i) issue_q1(i);
    issue_advance();
  };

  // ---- fragment geometry -------------------------------------------------------
  // v_mfma_f32_16x16x32_bf16: lane l holds row l % 16 of a 16-row block and 8
  // consecutive k, chosen by l / 16.  The four chunks of a stage's step t are
  // t, 2 + t, 4 + t and 6 + t, the same for both operands: with neighbouring
  // chunks (4 t + l / 16) the reads of 16 rows meet on the same LDS banks
  // (measured 300 B/ns per CU against 555, as the 32-row reads).
  // (The 32x32x16 form moves twice the accumulators per flop and runs at a
  // lower clock: the k loop alone, fragment reads included, on random operands
  // 1565 TFLOP/s against 1750; a second measurement of the latter 1629-1715.)
  const int r16 = l & 15;
  const int g4 = l >> 4;
  const int fa = cswz(r16);
  // First row of weight block pb of the wave.  SWIGLU: blocks 0, 1 are gate
  // rows, 2, 3 the matching up rows.
  const int arow0 = (EPI == EPI_SWIGLU ? 32 : 64) * wp;
  auto arow = [&](int pb) { return arow0 + (EPI == EPI_SWIGLU ? 16 * (pb & 1) + 128 * (pb >> 1) : 16 * pb); };
  // Fragment addresses: the chunk permutation cswz(row) & 7 of row 16 m + r16
  // is fa ^ 2 m, so k32 step, weight block and token block are compile-time
  // bits XORed into one lane register per operand, rebased per stage (held
  // per chunk and buffer the addresses would not fit beside the accumulators).
  const int lane_p = PT ? 0 : (arow0 + r16) * ROW_BYTES + (((2 * g4) ^ fa ^ ((arow0 >> 3) & 7)) << 4);
  const int lane_q = P_BYTES + (16 * wq + r16) * ROW_BYTES + (((2 * g4) ^ fa ^ (2 * wq)) << 4);
  // PT: lane l of 16-lane group g4 loads row 16 g4 + 8 t + 4 h + (l & 15) / 4
  // (h = 0, 1: the two halves of its 8 reduction values), columns
  // arow(pb) + 4 (l & 3) .. + 3; t and h do not enter ptswz of that row.
  const int tr_row = 16 * g4 + ((l & 15) >> 2);
  const int tr_base = tr_row * (TP * 2) + ((l & 1) << 3);
  const int tr_chunk = ((l & 2) >> 1) ^ ptswz(tr_row) ^ (8 * wp);  // arow0 = 64 wp: 8 chunks
  auto stage_base = [&](int lane, int s) {
    int v = lane;
    asm volatile("" : "+v"(v));  // (kept from being expanded outside the stage)
    return v + (s & 1) * STAGE_BYTES;
  };
  // Weight fragments of k32 step t.
  auto read_p = [&](bf16x8_t (&f)[NPB], int s, int t) {
    if constexpr (PT) {
      const int tb = stage_base(tr_base, s);
#pragma unroll
      for (int pb = 0; pb < NPB; ++pb) {
        const int off = tb + ((tr_chunk ^ (2 * pb)) << 4);
        short4_t v[2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
          v[h] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t*)(smem + off + (8 * t + 4 * h) * (TP * 2)));
        f[pb] = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(v[0], v[1], 0, 1, 2, 3, 4, 5, 6, 7));
      }
    } else {
      const int base = stage_base(lane_p, s);
#pragma unroll
      for (int pb = 0; pb < NPB; ++pb) {
        const int m = EPI == EPI_SWIGLU ? pb & 1 : pb;  // 16-row step inside the wave's rows
        f[pb] = *(const bf16x8_t*)(smem + (base ^ (t << 4) ^ ((2 * m) << 4)) + (arow(pb) - arow0) * ROW_BYTES);
      }
    }
  };
  // Token fragments of the wave's block j (tile rows 32 j + 16 wq .. + 15).
  auto read_q = [&](bf16x8_t (&f)[2], int base, int j) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
      f[t] = *(const bf16x8_t*)(smem + (base ^ (t << 4) ^ ((4 * (j & 1)) << 4)) + j * 32 * ROW_BYTES);
  };

  // ---- prologue: stages 0 and 1 in flight, stage 0 landed -----------------------
  // (the token-row DMA count of a stage depends on its tile's height, so the
  // wait is for everything issued)
  if constexpr (GATHER) {
    load_ids(0);
    wait_vm_barrier<0>();
  }
  issue_all(0);
  issue_all(1);
  wait_vm_barrier<DMA_P + QA>();

  int s = 0;
  // nks: the unit's k stages (ksteps for a whole tile); piece: the unit is
  // a piece of a split leftover tile.
  auto run_tile = [&](auto njv, int r, int row0, int row1, int pt, int nks, bool piece) {
    constexpr int NJV = decltype(njv)::value;
    constexpr int NU = NJV;
    floatx4_t acc[NPB][NJV];
#pragma unroll
    for (int i = 0; i < NPB; ++i)
#pragma unroll
      for (int j = 0; j < NJV; ++j) acc[i][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    // One stage, token block by token block (a unit: 8 MFMAs).  The wave holds
    // the stage's weight fragments (2 k32 steps) and reads the token
    // fragments two units ahead.
    //   A (before unit 2): every wave has read the stage's weight rows and
    //     its first four token blocks (tile rows 0..127), so the
    //     next-but-one stage's weight rows and first QA token-row
    //     instructions go into their place, spread over the following units
    //     (a burst of all of them stalls every wave's MFMAs behind the CU's
    //     address unit): they are in flight for almost two stages.
    //   B (before the last two units): every wave has read the whole stage;
    //     the rest of the next-but-one stage's token rows follow.  The wait
    //     there is for the next stage, i.e. for all but the DMA_P + QA
    //     instructions issued at A.
    // The last two units run after B while the next stage's first fragments
    // are read.
    bf16x8_t fp[2][NPB], fq[3][2];
    // DMA instruction d of the stage being issued: weight rows, then token rows
    auto issue_d = [&](auto dc) {
      constexpr int d = decltype(dc)::value;
      if constexpr (d < DMA_P)
        issue_p1(d);
      else
        issue_q1(d - DMA_P);
    };
    auto mfma_t = [&](int j, const bf16x8_t& q, int t) {
#pragma unroll
      for (int pb = 0; pb < NPB; ++pb)
        acc[pb][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fp[t][pb], q, acc[pb][j], 0, 0, 0);
    };
#pragma unroll
    for (int t = 0; t < 2; ++t) read_p(fp[t], s, t);
    read_q(fq[0], stage_base(lane_q, s), 0);
    if constexpr (NU > 1) read_q(fq[1], stage_base(lane_q, s), 1);
    auto stage = [&](auto lastc) {
      constexpr bool LAST = decltype(lastc)::value;
      constexpr int NA = DMA_P + QA, ND = DMA_P + DMA_Q;
      constexpr int UB = NU > 2 ? NU - 2 : 0, UA = UB < 2 ? UB : 2;
      constexpr int SPAN = UB > UA ? UB - UA : 1;
      bf16x8_t nq[2][2];
      const int qb = stage_base(lane_q, s);
      static_for<0, UB>([&](auto uc) {
        constexpr int u = decltype(uc)::value;
        if constexpr (u == UA) {
          lds_barrier();
          issue_prep(s + 2);
        }
        read_q(fq[(u + 2) % 3], qb, u + 2);
        if constexpr (u >= UA) static_for<NA * (u - UA) / SPAN, NA * (u - UA + 1) / SPAN>(issue_d);
        mfma_t(u, fq[u % 3][0], 0);
        mfma_t(u, fq[u % 3][1], 1);
        __builtin_amdgcn_sched_barrier(0);
      });
      if constexpr (UA == UB) {
        lds_barrier();
        issue_prep(s + 2);
        static_for<0, NA>(issue_d);
      }
      // the last units (one if the tile has one block), k32 step by step, so
      // that the next stage's weight fragments can be read in between
      wait_vm_barrier<NA>();
      const int qbn = LAST ? 0 : stage_base(lane_q, s + 1);
      static_for<0, 2>([&](auto tc) {
        constexpr int t = decltype(tc)::value;
        static_for<NA + (ND - NA) * t / 2, NA + (ND - NA) * (t + 1) / 2>(issue_d);
        if constexpr (!LAST && t < NU) read_q(nq[t], qbn, t);
        static_for<UB, NU>([&](auto uc) {
          constexpr int u = decltype(uc)::value;
          mfma_t(u, fq[u % 3][t], t);
        });
        if constexpr (!LAST) read_p(fp[t], s + 1, t);
        __builtin_amdgcn_sched_barrier(0);
      });
      issue_advance();
      if constexpr (!LAST) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          fq[0][i] = nq[0][i];
          if constexpr (NU > 1) fq[1][i] = nq[1][i];
        }
      }
      ++s;
    };
    for (int ks = 0; ks + 1 < nks; ++ks) stage(std::false_type{});
    stage(std::true_type{});

    // ---- split leftover tile: publish this piece's sums; the last piece
    //      to arrive adds all of them in piece order (the same order
    //      whichever arrives last) and runs the epilogue.  The partials are
    //      written back from this XCD's L2 (release) before the arrival is
    //      counted, and the last piece invalidates its caches (acquire)
    //      before it reads the others'.  The counter is reset for the next
    //      GEMM on this plan.
    if (__builtin_expect(piece, 0)) {  // (laid out away from the tile path)
      // Partial sums of leftover tile pc_t: np * kSplitPartBytes bytes at
      // part + pc_t * np * kSplitPartBytes, wave w's share (NPB * NJ blocks
      // of 1 KB per piece) at w * np * NPB * NJ KB, laid out block-major, then
      // piece (lane l: 16 bytes at 16 l).  The last piece then reads one
      // contiguous stream per wave: 1 KB chunk i is block i / np, piece i % np.
      // The bases are made opaque here so that no address is computed (and
      // kept live) in the k loop.
      constexpr uint32_t BLK = 1024;
      // (re-read here rather than held through the k loop)
      int info = pc_info;
      asm volatile("" : "+s"(info));
      const int np = info & 0xff, pc_j = (info >> 8) & 0xff, pc_t = info >> 16;
      const int4 pc = sload_int4((const int4*)((const char*)__builtin_amdgcn_kernarg_segment_ptr() +
                                               offsetof(FwdArgs, part)));
      float* const part = (float*)(((uint64_t)(uint32_t)pc.y << 32) | (uint32_t)pc.x);
      // (global address space: global rather than flat atomics and stores)
      gint_t* const split_cnt = (gint_t*)(((uint64_t)(uint32_t)pc.w << 32) | (uint32_t)pc.z);
      uint64_t pw = (uint64_t)part + (uint64_t)pc_t * np * kSplitPartBytes + (uint64_t)w * np * (NPB * NJ * BLK);
      asm volatile("" : "+s"(pw));
      // the lane id re-derived here (mbcnt of an opaque zero, which the
      // compiler cannot hoist), not kept through the k loop
      uint32_t zero = 0;
      asm volatile("" : "+v"(zero));
      uint32_t loff = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, zero)) * 16u;
      asm volatile("" : "+v"(loff));
      const uint32_t bstride = (uint32_t)np * BLK;  // one block of every piece
#pragma unroll
      for (int pb = 0; pb < NPB; ++pb)
#pragma unroll
        for (int j = 0; j < NJV; ++j) {
          const uint64_t dst = pw + (uint64_t)((pb * NJV + j) * bstride + pc_j * BLK);
          *(gfloatx4_t*)(dst + loff) = acc[pb][j];
        }
      wait_vm<0>();  // this wave's partial has reached L2
      __syncthreads();
      int* flag = (int*)(smem + FLAG_OFF);
      if (w == 0) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        int old = 0;
        if (l == 0) old = __hip_atomic_fetch_add(split_cnt + pc_t, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        old = __builtin_amdgcn_readfirstlane(old);
        if (old == np - 1) {
          if (l == 0) __hip_atomic_store(split_cnt + pc_t, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
          // the cache invalidation has completed before the barrier below
          // lets the other waves load the partials
          wait_vm<0>();
        }
        if (l == 0) *flag = (old == np - 1);
      }
      __syncthreads();
      if (__builtin_amdgcn_readfirstlane(*flag) == 0) return;
      // The sum in piece order.  Each wave streams its share through a ring
      // of 16 one-KB LDS slots (the free stage buffers) with LDS DMA, 16 KB
      // in flight and no VGPRs held for it: chunk i goes to slot i % 16, and
      // exactly one DMA is issued per chunk consumed (past the end: the last
      // chunk again, into the slot just read), so "at most 15 in flight"
      // means chunk i has landed.
      {
#pragma unroll
        for (int pb = 0; pb < NPB; ++pb)
#pragma unroll
          for (int j = 0; j < NJV; ++j) acc[pb][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
        constexpr int RING = 16;
        const int last = NPB * NJV * np - 1;
        const uint32_t ring = lds0 + (uint32_t)w * (RING * 1024);
        auto fetch = [&](int i) {
          dma16(loff, pw + (uint32_t)min(i, last) * 1024u, ring + (uint32_t)(i & (RING - 1)) * 1024u);
        };
#pragma unroll
        for (int i = 0; i < RING; ++i) fetch(i);
        const char* rbase = smem + w * (RING * 1024) + 16 * l;
        int i = 0;
#pragma unroll
        for (int pb = 0; pb < NPB; ++pb)
#pragma unroll
          for (int j = 0; j < NJV; ++j)
            for (int q = 0; q < np; ++q) {
              wait_vm<RING - 1>();
              acc[pb][j] += *(const floatx4_t*)(rbase + (i & (RING - 1)) * 1024);
              fetch(i + RING);  // after the adds: the slot's read has completed
              ++i;
            }
        wait_vm<0>();
      }
    }

    // ---- epilogue: acc[pb][j][i] is (token row 32 j + 16 wq + r16, weight
    //      row arow(pb) + 4 g4 + i).  Column validity is uniform over a block
    //      (H % 64 == 0 and N % 128 == 0 are required), row validity is per
    //      lane.  The scheduling barriers keep each block's accumulator reads
    //      next to their use (no 256-register hoist).  The lane's row and
    //      column group are re-materialised here (opaque copies) so that the
    //      compiler does not keep per-block offsets live across the k loop,
    //      where every register is taken.
    int er16 = r16;
    asm volatile("" : "+v"(er16));
    int eg4 = g4;
    asm volatile("" : "+v"(eg4));
    // A lane holds 4 consecutive columns (4 g4 ..) of each block.  For a pair
    // of neighbouring blocks (p, p + 1), v_permlane16_swap exchanges the odd
    // 16-lane rows of the first with the even rows of the second: lanes of
    // group g4 then hold columns 8 (g4 / 2) .. + 7 of block p + (g4 & 1), one
    // 16-byte store each.
    auto pair16 = [&](const uint32_t (&p0)[2], const uint32_t (&p1)[2]) {
      uint32_t x[2], y[2];
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        const auto sw = __builtin_amdgcn_permlane16_swap(p0[d], p1[d], false, false);
        x[d] = sw[0];
        y[d] = sw[1];
      }
      return u32x4_t{x[0], x[1], y[0], y[1]};
    };
    const int pcol = 16 * (eg4 & 1) + 8 * (eg4 >> 1);  // the lane's columns in a block pair
    // EPI_SWIGLU_BWD: saved pre-activation of token block jj
    auto load_h = [&](int jj, uint2 (&dst)[NPB][2]) {
      if constexpr (EPI == EPI_SWIGLU_BWD) {
        const int qrow = min(row0 + 32 * jj + 16 * wq + er16, row1 - 1);
#pragma unroll
        for (int pb = 0; pb < NPB; ++pb) {
          const int col = min(pt * TP + arow(pb), a.n_p - 16) + 4 * eg4;
          const bf16_t* hrow = a.h_in + (int64_t)qrow * a.ldh + col;
          dst[pb][0] = *(const uint2*)hrow;
          dst[pb][1] = *(const uint2*)(hrow + a.hidden);
        }
      }
    };
    // EPI_SWIGLU_BWD: the h values of token block j are loaded one block
    // ahead, into the other half of hbuf (double buffer).
    uint2 hbuf[2][NPB][2];
    if constexpr (EPI == EPI_SWIGLU_BWD) load_h(0, hbuf[0]);
#pragma unroll
    for (int j = 0; j < NJV; ++j) {
      const int trow = 32 * j + 16 * wq + er16;
      const int gq = row0 + trow;
      const bool row_ok = gq < row1;
      if constexpr (EPI == EPI_SWIGLU) {
        const float L = a.limit;
        // The clamp (swiglu_limit) is wave-uniform: one code path each, so
        // that the unclamped SwiGLU carries no min / max / select per value.
        // Gate and up are rounded to bf16 two at a time (one two-wide
        // conversion each; the bf16 pairs are what h_out stores).
        auto swiglu_rows = [&](auto clampc) {
          constexpr bool CLAMP = decltype(clampc)::value;
          uint32_t ap[2][2], gp[2][2], up[2][2];
#pragma unroll
          for (int pb = 0; pb < 2; ++pb) {
#pragma unroll
            for (int i2 = 0; i2 < 2; ++i2) {
              // h is materialised in bf16 by the reference; SwiGLU reads it.
              gp[pb][i2] = pack_bf16x2(acc[pb][j][2 * i2], acc[pb][j][2 * i2 + 1]);
              up[pb][i2] = pack_bf16x2(acc[pb + 2][j][2 * i2], acc[pb + 2][j][2 * i2 + 1]);
              float av[2];
#pragma unroll
              for (int h2 = 0; h2 < 2; ++h2) {
                float gc = __uint_as_float(h2 ? (gp[pb][i2] & 0xffff0000u) : (gp[pb][i2] << 16));
                float uc = __uint_as_float(h2 ? (up[pb][i2] & 0xffff0000u) : (up[pb][i2] << 16));
                if constexpr (CLAMP) {
                  gc = clamp_max_nan(gc, L);
                  uc = clamp_nan(uc, L);
                }
                av[h2] = silu_f(gc) * uc;
              }
              ap[pb][i2] = pack_bf16x2(av[0], av[1]);
            }
          }
          const u32x4_t av4 = pair16(ap[0], ap[1]);
          const int col = pt * 128 + 32 * wp + pcol;
          if (row_ok) *(u32x4_t*)(a.out + (int64_t)gq * a.ldo + col) = av4;
          if (a.h_out) {
            const u32x4_t gv4 = pair16(gp[0], gp[1]), uv4 = pair16(up[0], up[1]);
            if (row_ok) {
              bf16_t* hrow = a.h_out + (int64_t)gq * a.ldh + col;
              *(u32x4_t*)hrow = gv4;
              *(u32x4_t*)(hrow + a.hidden) = uv4;
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        };
        if (pt * 128 + 32 * wp < a.n_p) {
          if (a.limit == a.limit)
            swiglu_rows(std::true_type{});
          else
            swiglu_rows(std::false_type{});
        }
      } else if constexpr (EPI == EPI_SWIGLU_BWD) {
        // acc = dA = g for output columns p of the activation; with the saved
        // bf16 pre-activation h = [gate | up]: dgate, dup (clamp masks from
        // the bf16 h, as the reference's autograd sees them).
        // Without a clamp the limit is +inf: minimum / maximum against it are
        // exact no-ops (NaN included) and the masks are forced true, so the
        // value loop has no branch on the clamp.
        const bool noclamp = !(a.limit == a.limit);
        const float L = noclamp ? __builtin_inff() : a.limit;
        if (j + 1 < NJV) load_h(j + 1, hbuf[(j + 1) & 1]);
        const uint2 (&hv)[NPB][2] = hbuf[j & 1];
#pragma unroll
        for (int pp = 0; pp < NPB; pp += 2) {
          uint32_t dgp[2][2], dup[2][2], avp[2][2];
#pragma unroll
          for (int b2 = 0; b2 < 2; ++b2) {
            const int pb = pp + b2;
            const uint2 hg = hv[pb][0];
            const uint2 hu = hv[pb][1];
            const float gate[4] = {bf16_to_f32(hg.x & 0xffff), bf16_to_f32(hg.x >> 16), bf16_to_f32(hg.y & 0xffff),
                                   bf16_to_f32(hg.y >> 16)};
            const float up[4] = {bf16_to_f32(hu.x & 0xffff), bf16_to_f32(hu.x >> 16), bf16_to_f32(hu.y & 0xffff),
                                 bf16_to_f32(hu.y >> 16)};
            float dg[4], du[4], av[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const float gd = acc[pb][j][i];
              float gc = gate[i], uc = up[i];
              // torch.clamp's backward: where(in range, grad, 0), so exactly
              // zero where it clamped and where h is NaN
              const bool kg = noclamp | (gc <= L);
              const bool ku = noclamp | ((uc >= -L) & (uc <= L));
              gc = clamp_max_nan(gc, L);
              uc = clamp_nan(uc, L);
              const float sig = sigmoid_f(gc);
              const float sv = gc * sig;
              const float ds = sig * (1.f + gc * (1.f - sig));
              dg[i] = kg ? gd * uc * ds : 0.f;
              du[i] = ku ? gd * sv : 0.f;
              av[i] = sv * uc;
            }
#pragma unroll
            for (int d = 0; d < 2; ++d) {
              dgp[b2][d] = pack_bf16x2(dg[2 * d], dg[2 * d + 1]);
              dup[b2][d] = pack_bf16x2(du[2 * d], du[2 * d + 1]);
              avp[b2][d] = pack_bf16x2(av[2 * d], av[2 * d + 1]);
            }
            __builtin_amdgcn_sched_barrier(0);
          }
          const u32x4_t dg4 = pair16(dgp[0], dgp[1]), du4 = pair16(dup[0], dup[1]);
          const int col0 = pt * TP + arow(pp) + pcol;
          if (pt * TP + arow(pp) < a.n_p && row_ok) {
            bf16_t* drow = a.out + (int64_t)gq * a.ldo + col0;
            *(u32x4_t*)drow = dg4;
            *(u32x4_t*)(drow + a.hidden) = du4;
          }
          if (a.a_out) {
            const u32x4_t av4 = pair16(avp[0], avp[1]);
            if (pt * TP + arow(pp) < a.n_p && row_ok) *(u32x4_t*)(a.a_out + (int64_t)gq * a.hidden + col0) = av4;
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
        float sc = 1.f;
        int orow_idx = gq;
        if constexpr (EPI == EPI_SCATTER) {
          const int* meta = (const int*)(smem + LDS_BYTES + (r % 3) * META_BYTES);
          if (a.dest) orow_idx = min(max(meta[trow], 0), a.n_dest - 1);
          if (a.row_scale) {
            sc = __int_as_float(meta[TQ + trow]);
            if (a.scale_sigmoid) sc = sigmoid_f(sc);
          }
        }
        bf16_t* orow = a.out + (int64_t)orow_idx * a.ldo;
#pragma unroll
        for (int pp = 0; pp < NPB; pp += 2) {
          if (pt * TP + arow(pp) < a.n_p) {
            uint32_t pk[2][2];
#pragma unroll
            for (int b2 = 0; b2 < 2; ++b2) {
              const floatx4_t& v = acc[pp + b2][j];
              pk[b2][0] = pack_bf16x2(v[0] * sc, v[1] * sc);
              pk[b2][1] = pack_bf16x2(v[2] * sc, v[3] * sc);
            }
            const u32x4_t val = pair16(pk[0], pk[1]);
            const int col = pt * TP + arow(pp) + pcol;
            if (row_ok) {
              if (a.accumulate) {
                // add to the row already there (bf16 + bf16, one rounding)
                const u32x4_t prev = *(const u32x4_t*)(orow + col);
                u32x4_t sum;
#pragma unroll
                for (int d = 0; d < 4; ++d)
                  sum[d] = pack_bf16x2(bf16_to_f32(val[d] & 0xffffu) + bf16_to_f32(prev[d] & 0xffffu),
                                       bf16_to_f32(val[d] >> 16) + bf16_to_f32(prev[d] >> 16));
                *(u32x4_t*)(orow + col) = sum;
              } else {
                *(u32x4_t*)(orow + col) = val;
              }
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  };

  for (int r = 0; r < nmy; ++r) {
    const int tile = tile_at(r);
    const int qt = tile / a.np_tiles;
    const int pt = tile - qt * a.np_tiles;
    const int4 ti = sload_int4(a.table + qt);
    // 32-row blocks of the tile (at most TQ / 32): each token-row wave takes
    // 16 rows of every block
    const int nj = min((ti.z - ti.y + 31) >> 5, NJ);
    const bool piece = r >= nfull;
    const int nks = piece ? pc_k1 - pc_k0 : ksteps;
    switch (nj) {
      case 10: run_tile(std::integral_constant<int, 10>{}, r, ti.y, ti.z, pt, nks, piece); break;
      case 9: run_tile(std::integral_constant<int, 9>{}, r, ti.y, ti.z, pt, nks, piece); break;
      case 8: run_tile(std::integral_constant<int, 8>{}, r, ti.y, ti.z, pt, nks, piece); break;
      case 7: run_tile(std::integral_constant<int, 7>{}, r, ti.y, ti.z, pt, nks, piece); break;
      case 6: run_tile(std::integral_constant<int, 6>{}, r, ti.y, ti.z, pt, nks, piece); break;
      case 5: run_tile(std::integral_constant<int, 5>{}, r, ti.y, ti.z, pt, nks, piece); break;
      case 4: run_tile(std::integral_constant<int, 4>{}, r, ti.y, ti.z, pt, nks, piece); break;
      case 3: run_tile(std::integral_constant<int, 3>{}, r, ti.y, ti.z, pt, nks, piece); break;
      case 2: run_tile(std::integral_constant<int, 2>{}, r, ti.y, ti.z, pt, nks, piece); break;
      default: run_tile(std::integral_constant<int, 1>{}, r, ti.y, ti.z, pt, nks, piece); break;
    }
  }
  wait_vm<0>();  // DMAs past the end have landed before the workgroup exits
}

template <int EPI, bool PT = false, bool GATHER = false>
hipError_t launch_fwd(FwdArgs a, hipStream_t stream) {
  // set once per process (thread-safe static initialisation)
  static const hipError_t attr_err =
      hipFuncSetAttribute((const void*)gg_fwd_kernel<EPI, PT, GATHER>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS_TOTAL);
  if (attr_err != hipSuccess) return attr_err;
  const int grid = (num_cus() + 7) & ~7;
  return launch_k(true, gg_fwd_kernel<EPI, PT, GATHER>, dim3(grid), dim3(FTHREADS), LDS_TOTAL, stream, a);
}

}  // namespace

// Pieces per split leftover tile at most (TTAMD_GEMM_SPLIT=1 turns the
// split off, for A/B timing).
int split_max() {
  static const int v = [] {
    const char* e = getenv("TTAMD_GEMM_SPLIT");
    const int n = e ? atoi(e) : kSplitMaxPieces;
    return n < 1 ? 1 : (n > kSplitMaxPieces ? kSplitMaxPieces : n);
  }();
  return v;
}

// CUs of the device current at the first call (thread-safe static
// initialisation; every device of a process is the same part).
int num_cus() {
  static const int cus = [] {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    return n;
  }();
  return cus;
}

hipError_t launch_fwd_gemm(int epi, const FwdGemm& g, int small_rows, int small_cols, hipStream_t stream) {
  FwdArgs a = {};
  a.q = (const bf16_t*)g.act;
  a.ldq = g.kred;
  a.q_index = g.act_index;
  a.q_div = g.act_div > 0 ? g.act_div : 1;
  a.n_q_in = g.n_act;
  a.p = (const bf16_t*)g.w;
  a.kred = g.kred;
  a.ldp = g.kred;
  a.table = g.table;
  a.n_qtiles = g.n_qtiles;
  a.part = g.part;
  a.split_cnt = g.split_cnt;
  a.split_max = split_max();
  a.out = (bf16_t*)g.out;
  if (epi == EPI_SWIGLU) {
    a.p_estride = (int64_t)2 * g.n * g.kred;
    a.n_p = g.n;
    a.np_tiles = (g.n + 127) / 128;
    a.ldo = g.n;
    a.hidden = g.n;
    a.limit = g.limit;
    a.h_out = (bf16_t*)g.h_out;
    a.ldh = 2 * (int64_t)g.n;
    if (small_cols) return launch_small_gemm(epi, a, small_rows, small_cols, stream);
    if (a.q_index) return launch_fwd<EPI_SWIGLU, false, true>(a, stream);
    return launch_fwd<EPI_SWIGLU>(a, stream);
  }
  a.p_estride = (int64_t)g.n * g.kred;
  a.n_p = g.n;
  a.np_tiles = (g.n + TP - 1) / TP;
  a.ldo = g.n;
  a.row_scale = g.row_scale;
  a.dest = g.dest;
  a.n_dest = g.n_dest;
  a.accumulate = g.accumulate;
  a.scale_sigmoid = g.scale_sigmoid;
  if (small_cols) return launch_small_gemm(epi, a, small_rows, small_cols, stream);
  if (epi == EPI_SCATTER) return launch_fwd<EPI_SCATTER>(a, stream);
  return launch_fwd<EPI_STORE>(a, stream);
}

hipError_t launch_dgrad_gemm(int epi, const DgradGemm& g, hipStream_t stream) {
  // out[m, k] = sum_n dy[m, n] w[e, n, k]: token rows q = dy (reduction n
  // contiguous), weight operand w[e] = [n][k] reduction-major.
  FwdArgs a = {};
  a.q = (const bf16_t*)g.dy;
  a.ldq = g.n_red;
  a.q_div = 1;
  a.p = (const bf16_t*)g.w;
  a.p_estride = (int64_t)g.n_red * g.n_out;
  a.ldp = g.n_out;
  a.kred = g.n_red;
  a.n_p = g.n_out;
  a.np_tiles = (g.n_out + TP - 1) / TP;
  a.table = g.table;
  a.n_qtiles = g.n_qtiles;
  a.part = g.part;
  a.split_cnt = g.split_cnt;
  a.split_max = split_max();
  a.out = (bf16_t*)g.out;
  if (epi == EPI_SWIGLU_BWD) {
    a.ldo = 2 * (int64_t)g.n_out;
    a.hidden = g.n_out;
    a.limit = g.limit;
    a.h_in = (const bf16_t*)g.h;
    a.ldh = 2 * (int64_t)g.n_out;
    a.a_out = (bf16_t*)g.a_out;
    return launch_fwd<EPI_SWIGLU_BWD, true>(a, stream);
  }
  a.ldo = g.n_out;
  return launch_fwd<EPI_STORE, true>(a, stream);
}

}  // namespace ttamd
