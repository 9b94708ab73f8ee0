// Persistent grouped weight gradient on MI355X (gfx950):
//
//   dw[e][n][k] = sum_{m in rows(e)} dy[m][n] * x[m][k]
//
// The backward of torch._grouped_mm w.r.t. its weight (npu_gmm.py:31, :38
// under autograd): dw13 = dh^T x, dw2 = dy^T a per expert, reduction over the
// expert's ragged row range.
//
// Both operands are reduction-major (rows m, columns contiguous), so the
// MFMA fragments (8 consecutive m per lane) come from ds_read_b64_tr_b16 on
// the rows exactly as they arrive from HBM:
//   * Tile: 256 output rows n (the MFMA B operand, one n per lane) x 256
//     output columns k (A operand, 4 consecutive k per lane and register
//     group, so fp32 / bf16 results leave as 16- / 8-byte stores).
//   * 8 waves (2 per SIMD), 2 (n) x 4 (k); each wave 128 n x 64 k =
//     4 x 8 accumulators of v_mfma_f32_16x16x32_bf16 (half the accumulator
//     traffic per flop of the 32x32x16 form and, under the clock that the
//     load leaves, a 4-12 % higher MFMA rate).
//   * Stages of 64 rows m: x rows (64 x 512 bytes) and dy rows (64 x 512
//     bytes) DMA'd by global_load_lds_dwordx4 into two 64 KB buffers, chunk
//     c of row m stored at c ^ ptswz(m) (conflict-free transposed reads).
//     As in gemm_fwd.hip a stage is worked off one 16-column dy block at a
//     time with all of its x fragments in registers: its x rows are free
//     early and the next-but-one stage's go out at once, one DMA between the
//     MFMAs of each block; its dy rows follow at the stage's end.
//     Measured against 32x32x16 MFMAs with both operands' DMAs in one burst
//     per stage (one box, bf16 gradients): C3 routed dW13 1604 -> 1476 us,
//     dW2 779 -> 726, shared dW13 1185 -> 1080, dW2 620 -> 564; C2 shapes
//     dW13 530 -> 479, dW2 267 -> 246.
//   * The last stage of an expert reads clamped rows past its end; their
//     products are removed by zeroing those rows in both operands' fragments.
//   * Persistent over (expert, n tile, k tile), expert-major, the n tiles in
//     strips of 4 with the k tile major inside a strip (see tile_of), with
//     the XCD-aware slot mapping of gemm_fwd.hip; the DMA stream runs over
//     the flattened (tile, stage) sequence, whose stage counts vary per
//     expert.
//     An expert without rows still takes one (fully masked) stage, so its
//     gradient tile is written as zeros.
//   * Tail split (as in gemm_fwd.hip): with a workspace, the tiles left over
//     after the last full round are cut along the expert's rows into pieces
//     of consecutive stages, run on the otherwise idle workgroups; each
//     piece writes its fp32 sums to the workspace and counts its arrival,
//     and the last to arrive adds all of them in piece order (the same sum
//     whichever arrives last) and runs the epilogue.
#include <type_traits>

#include "common.h"
#include "dma_asm.h"
#include "gemm_common.h"
#include "kernels.h"

namespace ttamd {
namespace {

using namespace dma;

constexpr int TQ = 256;  // n per tile
constexpr int TP = 256;  // k per tile
constexpr int TK = 64;   // rows m per stage
constexpr int WAVES = 8;
constexpr int WPN = 4;              // waves along k
constexpr int NJ = TQ / 16 / 2;     // 8 n blocks of 16 per wave
constexpr int NPB = TP / 16 / WPN;  // 4 k blocks of 16 per wave
constexpr int THREADS = 64 * WAVES;
constexpr int ROW_BYTES = 512;      // 256 bf16 columns of one row m
constexpr int OP_BYTES = TK * ROW_BYTES;  // 32 KB per operand and stage
constexpr int STAGE_BYTES = 2 * OP_BYTES;
constexpr int LDS_BYTES = 2 * STAGE_BYTES;  // 128 KB
constexpr int SLAB_BYTES = 32 * 128;        // per wave: one 32 x 64 bf16 output block
constexpr int LDS_TOTAL = LDS_BYTES + WAVES * SLAB_BYTES;  // 160 KB
constexpr int DMA_OP = OP_BYTES / 1024 / WAVES;  // 4 instructions per operand and wave
constexpr int DMA_PER_STAGE = 2 * DMA_OP;
constexpr int kStripN = 4;  // n tiles per strip of the tile order

typedef short short4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) short4_t lds_short4_t;
typedef __attribute__((address_space(1))) int gint_t;
typedef __attribute__((address_space(1))) floatx4_t gfloatx4_t;

// Chunk permutation of a row (as gemm_fwd.hip's reduction-major weights).
__device__ __forceinline__ int ptswz(int m) { return 2 * ((m & 3) | ((m >> 2) & 4)); }

// f(integral_constant) for A, A + 1, ..., B - 1.
template <int A, int B, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (A < B) {
    f(std::integral_constant<int, A>{});
    static_for<A + 1, B>(f);
  }
}

__global__ __launch_bounds__(THREADS, 1) void gg_wgrad_dma_kernel(const WgradDmaArgs a) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wq = w / WPN;
  const int wp = w % WPN;
  const int l = threadIdx.x & 63;
  const int G = gridDim.x;
  const int b = blockIdx.x;
  const int slot = (b & 7) * (G >> 3) + (b >> 3);
  const int per_e = a.n_tiles * a.k_tiles;
  const int ntiles = a.E * per_e;
  // Tail split: R full rounds, rt tiles left over; piece j of leftover tile
  // t runs on slot j * rt + t after the slot's R whole tiles.
  const int R = ntiles / G;
  const int rt = ntiles - R * G;
  const int np = (a.split_np > 1 && rt > 0 && rt <= kSplitTiles && a.split_np * rt <= G) ? a.split_np : 1;
  const bool has_piece = np > 1 && slot < rt * np;
  const int nfull = np > 1 ? R : (slot < ntiles ? (ntiles - slot + G - 1) / G : 0);
  const int nmy = nfull + (has_piece ? 1 : 0);
  if (nmy == 0) return;
  const int pc_t = has_piece ? slot % rt : 0;  // leftover tile of the piece
  const int pc_j = has_piece ? slot / rt : 0;  // piece index
  const uint32_t lds0 = lds_addr(smem);

  // tile round r -> (expert, n tile, k tile, first row, end row, stages)
  struct Tile {
    int e, nt, kt, m0, m1, nks;
  };
  auto tile_of = [&](int r) {
    Tile t;
    const int id = r < nfull ? r * G + slot : R * G + pc_t;
    t.e = id / per_e;
    const int rem = id - t.e * per_e;
    // Within an expert, strips of kStripN n tiles, k tile major inside a
    // strip: an XCD's 32 consecutive slots then cover 4 n x 8 k tiles, so
    // each dY slice is shared by 8 of its workgroups and each X slice by 4
    // in its L2 (row-major: one n tile x 32 k tiles, every X slice read by
    // one workgroup of the XCD).
    const int strip = rem / (kStripN * a.k_tiles);
    const int in_strip = rem - strip * kStripN * a.k_tiles;
    const int gn = min(kStripN, a.n_tiles - strip * kStripN);
    t.kt = in_strip / gn;
    t.nt = strip * kStripN + (in_strip - t.kt * gn);
    t.m0 = t.e == 0 ? 0 : sload_int(a.offs + t.e - 1);
    t.m1 = sload_int(a.offs + t.e);
    t.m0 = min(max(t.m0, 0), a.M);
    t.m1 = min(max(t.m1, t.m0), a.M);
    t.nks = max(1, (t.m1 - t.m0 + TK - 1) / TK);
    if (r >= nfull) {
      // piece pc_j: stages [k0, k1) of the tile's rows (an empty share runs
      // one fully masked stage and contributes zeros)
      const int k0 = pc_j * t.nks / np, k1 = (pc_j + 1) * t.nks / np;
      const int m_end = t.m1;
      t.m1 = min(t.m0 + TK * k1, m_end);
      t.m0 = min(t.m0 + TK * k0, m_end);
      t.nks = max(1, k1 - k0);
    }
    return t;
  };

  // ---- DMA stream: a cursor over (tile round, stage) --------------------------
  // instruction i of wave w moves rows 2 (WAVES i + w) and + 1 of an operand;
  // lane l: row + (l >> 5), physical chunk l & 31.  The chunk permutation
  // depends on i through bit 3 (i % 2) only; a tile with 128 valid columns
  // (N, K % 128 == 0) reads those twice.
  int c_r = 0, c_ks = 0;
  Tile c_t = tile_of(0);
  const int d_row = 2 * w + (l >> 5);
  const int d_chunk = (l & 31) ^ ptswz(d_row);
  uint64_t d_xb = 0, d_yb = 0;
  int d_mstage = 0, d_last = 0, d_xmask = 31, d_ymask = 31;
  uint32_t d_st = 0;
  // bases of the stage issued next, into the buffer of stage s
  auto issue_prep = [&](int s) {
    d_mstage = c_t.m0 + TK * c_ks;
    d_last = c_t.m1 - 1;  // below d_mstage for an expert without rows
    d_xb = (uint64_t)(a.x + (int64_t)c_t.kt * TP);
    d_yb = (uint64_t)(a.dy + (int64_t)c_t.nt * TQ);
    d_xmask = a.K - c_t.kt * TP >= TP ? 31 : 15;
    d_ymask = a.N - c_t.nt * TQ >= TQ ? 31 : 15;
    if (a.M == 0) {  // no rows at all: every stage is masked; any readable address will do
      d_xb = d_yb = (uint64_t)a.dw;
      d_xmask = d_ymask = 15;
    }
    d_st = lds0 + (uint32_t)((s & 1) * STAGE_BYTES) + w * 1024;
  };
  const int m_max = max(a.M - 1, 0);
  auto row_of = [&](int i) { return min(max(min(d_mstage + d_row + 2 * WAVES * i, d_last), 0), m_max); };
  auto issue_x = [&](int i) {
    const uint32_t voff = (uint32_t)row_of(i) * (uint32_t)(a.ldx * 2) + (((d_chunk ^ (8 * (i & 1))) & d_xmask) << 4);
    dma16(voff, d_xb, d_st + i * (WAVES * 1024));
  };
  auto issue_y = [&](int i) {
    const uint32_t voff = (uint32_t)row_of(i) * (uint32_t)(a.lddy * 2) + (((d_chunk ^ (8 * (i & 1))) & d_ymask) << 4);
    dma16(voff, d_yb, d_st + OP_BYTES + i * (WAVES * 1024));
  };
  // past the last stage keep re-loading it
  auto issue_advance = [&]() {
    if (c_ks + 1 < c_t.nks) {
      ++c_ks;
    } else if (c_r + 1 < nmy) {
      ++c_r;
      c_ks = 0;
      c_t = tile_of(c_r);
    }
  };

  // ---- fragments: transposed reads (see gemm_fwd.hip, PT) ---------------------
  // k32 step t: lane l of 16-lane group g4 holds rows 16 g4 + 8 t .. + 7 of
  // column col0 + l % 16, from two reads of rows + 4 h + (l & 15) / 4,
  // columns col0 + 4 (l & 3) .. + 3; t and h do not enter ptswz of the row.
  const int r16 = l & 15;
  const int g4 = l >> 4;
  const int tr_row = 16 * g4 + (r16 >> 2);
  // A block of 16 columns is two chunks: block m of the wave's columns and the
  // permutation only XOR bits 5..8 of the lane's address.
  const int tr_base = tr_row * ROW_BYTES + ((l & 1) << 3);
  const int tr_chunk = ((l & 2) >> 1) ^ ptswz(tr_row);
  const int arow0 = (TP / WPN) * wp, brow0 = (TQ / 2) * wq;
  const int lane_x = tr_base + ((tr_chunk ^ (arow0 >> 3)) << 4);
  const int lane_y = OP_BYTES + tr_base + ((tr_chunk ^ (brow0 >> 3)) << 4);
  auto stage_base = [&](int lane, int s) {
    int v = lane;
    asm volatile("" : "+v"(v));  // (kept from being expanded outside the stage)
    return v + (s & 1) * STAGE_BYTES;
  };
  auto tr8 = [&](int base, int m, int t) {
    const char* p = smem + (base ^ (m << 5)) + 8 * t * ROW_BYTES;
    short4_t v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t*)p);
    short4_t v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t*)(p + 4 * ROW_BYTES));
    return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  auto read_x = [&](bf16x8_t (&f)[NPB], int s, int t) {
    const int base = stage_base(lane_x, s);
#pragma unroll
    for (int pb = 0; pb < NPB; ++pb) f[pb] = tr8(base, pb, t);
  };
  auto read_y = [&](bf16x8_t (&f)[2], int base, int j) {
#pragma unroll
    for (int t = 0; t < 2; ++t) f[t] = tr8(base, j, t);
  };
  // Rows >= nvalid of a stage contribute nothing: zero them in both the x
  // and the dy fragments (the clamped rows loaded there belong to the same
  // or, for an expert without rows, the previous expert; zeroing only one
  // operand would turn an Inf or NaN there into NaN instead of the exact
  // zeros the gradient of an empty expert is).  Element i of the lane's 8 is
  // row 16 g4 + 8 t + i.
  auto mask = [&](bf16x8_t& f, int t, int nvalid) {
    const int rem = nvalid - 16 * g4 - 8 * t;
    u32x4_t v = __builtin_bit_cast(u32x4_t, f);
#pragma unroll
    for (int d = 0; d < 4; ++d) v[d] &= (2 * d < rem ? 0x0000ffffu : 0u) | (2 * d + 1 < rem ? 0xffff0000u : 0u);
    f = __builtin_bit_cast(bf16x8_t, v);
  };

  // ---- prologue --------------------------------------------------------------
#pragma unroll
  for (int st = 0; st < 2; ++st) {
    issue_prep(st);
#pragma unroll
    for (int i = 0; i < DMA_OP; ++i) issue_x(i);
#pragma unroll
    for (int i = 0; i < DMA_OP; ++i) issue_y(i);
    issue_advance();
  }
  wait_vm_barrier<DMA_PER_STAGE>();
  bf16x8_t fx[2][NPB], fy[4][2];  // dy block j in buffer j % 4
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    read_x(fx[t], 0, t);
    read_y(fy[t], stage_base(lane_y, 0), t);
  }

  int s = 0;
  for (int r = 0; r < nmy; ++r) {
    const Tile t = tile_of(r);
    floatx4_t acc[NPB][NJ];
#pragma unroll
    for (int i = 0; i < NPB; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    // One stage, dy block by dy block (8 MFMAs each), the dy fragments read
    // two blocks ahead.
    //   A (before block 2): every wave has read the stage's x rows; the
    //     next-but-one stage's go out, one instruction per block.
    //   B (before the last two blocks): every wave has read the whole stage
    //     and the next one has landed (all but the DMA_OP instructions
    //     issued at A); the next-but-one stage's dy rows follow.
    // The first and last two blocks run k32 step by k32 step, while the next
    // stage's first fragments are read.
    auto stage = [&](auto maskedc, int nvalid) {
      constexpr bool MASKED = decltype(maskedc)::value;
      auto mfma_t = [&](int j, int tt) {
        if constexpr (MASKED) mask(fy[j % 4][tt], tt, nvalid);
#pragma unroll
        for (int pb = 0; pb < NPB; ++pb)
          acc[pb][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fx[tt][pb], fy[j % 4][tt], acc[pb][j], 0, 0, 0);
      };
      const int yb = stage_base(lane_y, s);
      static_for<0, 2>([&](auto tc) {
        constexpr int tt = decltype(tc)::value;
        if constexpr (MASKED) {
#pragma unroll
          for (int pb = 0; pb < NPB; ++pb) mask(fx[tt][pb], tt, nvalid);
        }
        read_y(fy[tt + 2], yb, tt + 2);
        mfma_t(0, tt);
        mfma_t(1, tt);
        __builtin_amdgcn_sched_barrier(0);
      });
      lds_barrier();
      issue_prep(s + 2);
      static_for<2, NJ - 2>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        read_y(fy[(j + 2) % 4], yb, j + 2);
        issue_x(j - 2);
        mfma_t(j, 0);
        mfma_t(j, 1);
        __builtin_amdgcn_sched_barrier(0);
      });
      static_assert(NJ - 4 == DMA_OP, "one x instruction per block between the barriers");
      wait_vm_barrier<DMA_OP>();
      const int ybn = stage_base(lane_y, s + 1);
      static_for<0, 2>([&](auto tc) {
        constexpr int tt = decltype(tc)::value;
        read_y(fy[tt], ybn, tt);
        issue_y(2 * tt);
        mfma_t(NJ - 2, tt);
        issue_y(2 * tt + 1);
        mfma_t(NJ - 1, tt);
        __builtin_amdgcn_sched_barrier(0);
        read_x(fx[tt], s + 1, tt);
        __builtin_amdgcn_sched_barrier(0);
      });
      issue_advance();
      ++s;
    };
    // only a tile's last stage can be partial
    const int nvalid = t.m1 - t.m0 - TK * (t.nks - 1);
    for (int ks = nvalid < TK ? 1 : 0; ks < t.nks; ++ks) stage(std::false_type{}, TK);
    if (nvalid < TK) stage(std::true_type{}, nvalid);

    // ---- split leftover tile: publish this piece's sums; the last piece to
    //      arrive adds all of them in piece order and runs the epilogue.
    //      The partials are written back from this XCD's L2 (release) before
    //      the arrival is counted, and the last piece invalidates its caches
    //      (acquire) before it reads the others'; it resets the counter.
    if (np > 1 && r >= nfull) {
      constexpr int NV4 = NPB * NJ;                       // float4 per lane
      constexpr uint32_t WAVE_BYTES = NV4 * 64 * 16;      // 32 KB
      constexpr uint64_t PIECE_BYTES = (uint64_t)WAVES * WAVE_BYTES;  // 256 KB
      static_assert(PIECE_BYTES <= kSplitPartBytes, "partial of a piece");
      // The bases are made opaque here so that no address is computed (and
      // kept live) in the k loop.
      uint64_t pw = (uint64_t)a.part + (uint64_t)w * WAVE_BYTES;
      asm volatile("" : "+s"(pw));
      uint32_t loff = (uint32_t)l * 16u;
      asm volatile("" : "+v"(loff));
      auto piece = [&](int j) { return pw + (uint64_t)(pc_t * np + j) * PIECE_BYTES; };
      const uint64_t mine = piece(pc_j);
#pragma unroll
      for (int pb = 0; pb < NPB; ++pb)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          *(gfloatx4_t*)(mine + (uint32_t)((pb * NJ + j) * 1024) + loff) = acc[pb][j];
      wait_vm<0>();  // this wave's partial has reached L2; every DMA has landed
      __syncthreads();
      // (the stage buffers are idle: no DMA is issued after the last unit)
      int* flag = (int*)smem;
      if (w == 0) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        gint_t* cnt = (gint_t*)(a.split_cnt + pc_t);
        int old = 0;
        if (l == 0) old = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        old = __builtin_amdgcn_readfirstlane(old);
        if (old == np - 1) {
          if (l == 0) __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
          // the cache invalidation has completed before the barrier below
          // lets the other waves load the partials
          wait_vm<0>();
        }
        if (l == 0) *flag = (old == np - 1);
      }
      __syncthreads();
      if (__builtin_amdgcn_readfirstlane(*flag) == 0) return;
#pragma unroll
      for (int pb = 0; pb < NPB; ++pb)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[pb][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
      // the sum in piece order, four blocks (loads) at a time
      for (int jp = 0; jp < np; ++jp) {
        const uint64_t src = piece(jp);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          floatx4_t v[NPB];
#pragma unroll
          for (int pb = 0; pb < NPB; ++pb) v[pb] = *(const gfloatx4_t*)(src + (uint32_t)((pb * NJ + j) * 1024) + loff);
#pragma unroll
          for (int pb = 0; pb < NPB; ++pb) acc[pb][j] += v[pb];
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }

    // ---- epilogue: acc[pb][j][i] = dw[e][n][k], n = nt*TQ + brow0 + 16 j +
    //      lane % 16, k = kt*TP + arow0 + 16 pb + 4 (lane / 16) + i.
    int er16 = r16;
    asm volatile("" : "+v"(er16));
    // Both forms go through the wave's private 4 KB LDS slab (row r: 128
    // bytes, 16-byte chunk c at c ^ (r & 7)) and leave as streaming stores
    // of 8 whole 128-byte rows per instruction: the gradient is written once
    // and not read here again, and cached it would evict the operand lines
    // the other workgroups of the XCD are about to read (routed C3 dW2 934
    // -> 724 us in bf16).
    char* slab = smem + LDS_BYTES + w * SLAB_BYTES;
    if (a.dw_fp32) {
      // fp32: one 32-row x 32-column block (128 bytes per row) at a time
#pragma unroll
      for (int j = 0; j < NJ; j += 2) {
#pragma unroll
        for (int pb = 0; pb < NPB; pb += 2) {
          if (t.kt * TP + arow0 + 16 * pb < a.K) {  // wave-uniform: the block's 32 columns are valid together
#pragma unroll
            for (int jj = 0; jj < 2; ++jj)
#pragma unroll
              for (int p = 0; p < 2; ++p) {
                const int row = 16 * jj + er16, chunk = (4 * p + g4) ^ (er16 & 7);  // columns 16 p + 4 g4 .. + 3
                *(floatx4_t*)(slab + row * 128 + chunk * 16) = acc[pb + p][j + jj];
              }
            lds_wait();  // the slab writes have landed
            uint4 o4[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int r = 8 * i + (l >> 3);
              o4[i] = *(const uint4*)(slab + r * 128 + (((l & 7) ^ (r & 7)) << 4));
            }
            lds_wait();  // read before the next block overwrites the slab
            const int col = t.kt * TP + arow0 + 16 * pb + 4 * (l & 7);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int n = t.nt * TQ + brow0 + 16 * j + 8 * i + (l >> 3);
              if (n < a.N) store_stream((uint4*)((float*)a.dw + ((int64_t)t.e * a.N + n) * a.K + col), o4[i]);
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    } else if (t.kt * TP + arow0 < a.K) {  // the wave's 64 columns are valid together
      // bf16: one 32-row block (the wave's 64 columns, 128 bytes per row)
      // at a time
      const int col = t.kt * TP + arow0 + 8 * (l & 7);
#pragma unroll
      for (int j = 0; j < NJ; j += 2) {
#pragma unroll
        for (int jj = 0; jj < 2; ++jj)
#pragma unroll
          for (int pb = 0; pb < NPB; ++pb) {
            const floatx4_t& v = acc[pb][j + jj];
            const int row = 16 * jj + er16, chunk = (2 * pb + (g4 >> 1)) ^ (er16 & 7);
            *(uint2*)(slab + row * 128 + chunk * 16 + (g4 & 1) * 8) =
                make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
          }
        lds_wait();  // the slab writes have landed
        uint4 o4[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 8 * i + (l >> 3);
          o4[i] = *(const uint4*)(slab + r * 128 + (((l & 7) ^ (r & 7)) << 4));
        }
        lds_wait();  // read before the next block overwrites the slab
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int n = t.nt * TQ + brow0 + 16 * j + 8 * i + (l >> 3);
          if (n < a.N) store_stream((uint4*)((bf16_t*)a.dw + ((int64_t)t.e * a.N + n) * a.K + col), o4[i]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  wait_vm<0>();
}

// Arrival counters of the split tail tiles to zero (a kernel, not a memset,
// so that the sequence can be captured in a HIP graph).
__global__ __launch_bounds__(256) void split_cnt_zero_kernel(int* __restrict__ cnt, int n) {
  for (int i = threadIdx.x; i < n; i += 256) cnt[i] = 0;
}

}  // namespace

hipError_t launch_split_cnt_zero(int* split_cnt, int n, hipStream_t stream) {
  return launch_k(false, split_cnt_zero_kernel, dim3(1), dim3(256), 0, stream, split_cnt, n);
}

hipError_t launch_wgrad_dma(const WgradDmaArgs& a, hipStream_t stream) {
  // set once per process (thread-safe static initialisation)
  static const hipError_t attr_err =
      hipFuncSetAttribute((const void*)gg_wgrad_dma_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS_TOTAL);
  if (attr_err != hipSuccess) return attr_err;
  const int grid = (num_cus() + 7) & ~7;
  return launch_k(false, gg_wgrad_dma_kernel, dim3(grid), dim3(THREADS), LDS_TOTAL, stream, a);
}

}  // namespace ttamd
