// Grouped GEMM of the expert FFN forward for few rows per expert or few
// tiles (decode, short prefill, small models) on MI355X (gfx950).
//
//   out[q, p] = sum_k act[q, k] * w[e(q), p, k]        (k contiguous in both)
//
// With up to ~128 rows per expert the path is bound by streaming every hit
// expert's weights from HBM once, not by the MFMAs, and what the streaming
// rate needs is requests in flight all the time: a copy of the weight stream
// alone (LDS DMA, one workgroup per CU) reaches 6.1 TB/s with 64 KB in
// flight per CU and 4.7 with 32 KB.  The 320 x 256 kernel (gemm_fwd.hip) holds
// about one stage in flight across its barriers; with few tiles it leaves CUs
// idle, and every tile of few rows costs it the time of 160.
//
// Tile: up to TQ (64 or 128) token rows x STP (128 or 256) weight rows, k in
// stages of 64 (128-byte rows).  A ring of NS stages, one barrier per stage
// that waits for the oldest stage only (counted vmcnt) and issues the stage
// NS - 1 ahead into the buffer freed by the previous stage, so NS - 2 whole
// stages (40-96 KB) stay in flight across every barrier and the stream runs
// on through the epilogue into the next tile.  Every wave issues the same
// number of DMAs per stage (token rows past the tile repeat its last row),
// so the count is a constant.
//   64 x 128: 6 x 24 KB   few rows or few tiles: twice the tiles, so that a
//                         few experts still occupy every CU
//   64 x 256: 3 x 40 KB   half the token-row traffic per weight byte
//  128 x 128: 4 x 32 KB,  128 x 256: 3 x 48 KB   up to ~100 rows per expert
//
// 8 waves as 2 (token) x 4 (weight): wave (wq, wp) owns the 32-row weight
// blocks wp, wp + 4 and token blocks wq, wq + 2; accumulators of
// v_mfma_f32_32x32x16_bf16 with the weights as A.  SWIGLU: the tile's rows
// alternate in blocks of 8 between gate and up (STP / 2 columns of each), so
// a lane's accumulator groups g = 0, 2 are gate columns and g = 1, 3 the
// matching up columns, and the activation needs no exchange.
//
// Measured, w13 / w2, us, against the 320 x 256 kernel: 64 experts of 768 x
// 2048 (Qwen3-30B-A3B), 2 rows each 65 / 29 against 76 / 32, 64 rows 83 / 40
// against 92 / 40; 128 of them a tie from 2 to 40 rows (127 / 66 and 152 / 89
// against 129 / 69 and 147 / 88: 5.9-6.1 TB/s of weights on both); 32 of 7168
// x 2048, 9 rows 306 / 166 against 307 / 179; the 256 x 512 debug model's 2000
// rows 8 / 10 against 19 / 20 (32 and 8 large tiles on 256 CUs).  Against the
// large kernel with one stage barrier for everything in flight, both GEMMs and
// the K-way sum: 128 experts of 768 x 2048, 32 tokens 243 -> 196 us, 1003
// tokens 299 -> 251; the shard of 32, 200 rows 553 -> 470.
//
// Reference semantics: torchtitanturbo/models/common/npu_gmm.py:17-38.
#include "common.h"
#include "dma_asm.h"
#include "gemm_common.h"
#include "kernels.h"

namespace ttamd {
namespace {

using namespace dma;

constexpr int STK = 64;              // k per stage: 128-byte rows
constexpr int SWAVES = 8;
constexpr int SROW = STK * 2;
constexpr int META_SLOTS = 8;                     // EPI_SCATTER row metadata, tile round % 8

template <int TQ, int STP>
struct Geo {
  static constexpr int NS = STP == 256 ? 3 : TQ == 64 ? 6 : 4;
  static constexpr int SP_BYTES = STP * SROW;
  static constexpr int SDMA_P = STP / 8 / SWAVES;  // weight-row DMAs per wave and stage
  static constexpr int NPB = STP / 128;            // 32-row weight blocks per wave
  static constexpr int DMA_Q = TQ / 8 / SWAVES;
  static constexpr int IPW = SDMA_P + DMA_Q;  // DMAs per wave and stage
  static constexpr int NJ = TQ / 64;          // token blocks per wave
  static constexpr int STAGE = SP_BYTES + TQ * SROW;
  static constexpr int RING = NS * STAGE;  // 144 KB (64 x 128, 128 x 256), 120 KB (64 x 256), 128 KB (128 x 128)
  static constexpr int META = TQ * 8;      // destination rows, scales
  // gathered rows: per wave, two slots (tile round % 2) of DMA_Q x 64 ids
  static constexpr int IDS = SWAVES * 2 * DMA_Q * 256;
  static constexpr int EXTRA = META_SLOTS * META > IDS ? META_SLOTS * META : IDS;
  static constexpr int LDS = RING + EXTRA;
  static_assert(LDS <= 160 * 1024, "LDS of a CU");
};

template <int EPI, bool GATHER, int TQ, int STP>
__global__ __launch_bounds__(64 * SWAVES, 1) void gg_small_kernel(const FwdArgs a) {
  using L = Geo<TQ, STP>;
  constexpr int SP_BYTES = L::SP_BYTES, SDMA_P = L::SDMA_P, NPB = L::NPB;
  constexpr int COLS = EPI == EPI_SWIGLU ? STP / 2 : STP;  // output columns per tile
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wq = w >> 2;
  const int wp = w & 3;
  const int l = threadIdx.x & 63;
  const int G = gridDim.x;
  const int b = blockIdx.x;
  auto U = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
  const int nqt = sload_int(a.n_qtiles);
  const int ntiles = nqt * a.np_tiles;
  const int ksteps = U(a.kred / STK);
  // Full rounds: XCD x takes the consecutive tiles [x G/8, (x+1) G/8) of the
  // round (one expert's token rows and shared weight tiles in its L2).  The
  // last, partial round goes to the blocks in hardware order, which spreads
  // it over all eight XCDs.
  const int R = U(ntiles / G);
  const int rt = ntiles - R * G;
  const int slot = (b & 7) * (G >> 3) + (b >> 3);
  const int nmy = R + (b < rt ? 1 : 0);
  if (nmy == 0) return;
  const int total = nmy * ksteps;
  // Token tiles in pairs, weight tile major inside a pair: the two token
  // tiles of an expert share each weight tile while it is in the L2.
  auto tile_at = [&](int r, int& qt, int& pt) {
    const int t = r < R ? r * G + slot : R * G + b;
    const int blk = t / (2 * a.np_tiles);
    const int in_blk = t - blk * 2 * a.np_tiles;
    const int gq = min(2, nqt - 2 * blk);
    pt = in_blk / gq;
    qt = 2 * blk + (in_blk - pt * gq);
  };

  const uint32_t lds0 = lds_addr(smem);
  const int drow = l >> 3;
  const int rr0 = 8 * w + drow;  // row of DMA 0; DMA i moves rows rr0 + 64 i
  const uint32_t lch16 = (uint32_t)(((l & 7) ^ ((drow ^ w) & 7)) * 16);

  // ---- DMA stream -----------------------------------------------------------
  auto load_ids = [&](int r) {
    int qt, pt;
    tile_at(r, qt, pt);
    const int4 ti = sload_int4(a.table + qt);
#pragma unroll
    for (int i = 0; i < L::DMA_Q; ++i) {
      const uint32_t row = (uint32_t)min(rr0 + 64 * i, ti.z - ti.y - 1);
      dma4(row * 4, (uint64_t)(a.q_index + ti.y), lds0 + L::RING + (uint32_t)(((w * 2 + (r & 1)) * L::DMA_Q + i) * 256));
    }
  };
  int d_r = -1, d_rot = 0;
  uint64_t d_pbase = 0, d_qbase = 0;
  uint32_t d_poff[SDMA_P], d_qoff[L::DMA_Q];
  auto dma_tile = [&](int r) {
    int qt, pt;
    tile_at(r, qt, pt);
    const int4 ti = sload_int4(a.table + qt);
    const int qmax = ti.z - ti.y - 1;
#pragma unroll
    for (int i = 0; i < SDMA_P; ++i) {
      const int rb = SWAVES * i + w;  // 8-row block of the tile
      const int last = a.n_p - 1 - pt * COLS;
      const int row = EPI == EPI_SWIGLU ? (rb & 1 ? (int)a.hidden : 0) + min(8 * (rb >> 1) + drow, last)
                                        : min(8 * rb + drow, last);
      d_poff[i] = (uint32_t)row * (uint32_t)(a.ldp * 2) + lch16;
    }
    if constexpr (GATHER) {
      // ids of this tile: DMA'd while the previous tile was issued; with
      // few stages per tile that may still be in flight
      if (ksteps < L::NS) wait_vm<0>();
#pragma unroll
      for (int i = 0; i < L::DMA_Q; ++i) {
        const int* ids = (const int*)(smem + L::RING + ((w * 2 + (r & 1)) * L::DMA_Q + i) * 256);
        const int src = min(max(ids[l] / a.q_div, 0), a.n_q_in - 1);
        d_qoff[i] = (uint32_t)src * (uint32_t)(a.ldq * 2) + lch16;
      }
      if (r + 1 < nmy) load_ids(r + 1);
      d_qbase = (uint64_t)a.q;
    } else {
#pragma unroll
      for (int i = 0; i < L::DMA_Q; ++i)
        d_qoff[i] = (uint32_t)min(rr0 + 64 * i, qmax) * (uint32_t)(a.ldq * 2) + lch16;
      d_qbase = (uint64_t)(a.q + (int64_t)ti.y * a.ldq);
    }
    d_pbase = (uint64_t)(a.p + (int64_t)ti.x * a.p_estride +
                         (int64_t)pt * COLS * a.ldp);
    // Rows a multiple of 4 KB apart: the workgroups, all at the same k, would
    // ask the same HBM channels (5.1-5.6 TB/s); each weight tile starts its k
    // walk elsewhere (6.1).  Other row lengths spread by themselves.
    d_rot = (a.ldp * 2) % 4096 == 0 ? U((5 * pt + 3 * ti.x) % ksteps) : 0;
    if constexpr (EPI == EPI_SCATTER) {
      for (int c = w; c < TQ / 64; c += SWAVES) {
        const uint32_t q = (uint32_t)min(64 * c + l, qmax);
        const uint32_t m = lds0 + L::RING + (uint32_t)((r % META_SLOTS) * L::META) + c * 256;
        if (a.dest) dma4(q * 4, (uint64_t)(a.dest + ti.y), m);
        if (a.row_scale) dma4(q * 4, (uint64_t)(a.row_scale + ti.y), m + TQ * 4);
      }
    }
    d_r = r;
  };
  // Stages are issued in order 0, 1, 2, ...; past the end the last stage is
  // issued again (into its own ring slot, read by nobody).
  int n_r = 0, n_ks = 0, n_left = total, n_buf = 0;
  auto issue = [&]() {
    if (n_r != d_r) dma_tile(n_r);
    int ks = n_ks + d_rot;
    ks = ks >= ksteps ? ks - ksteps : ks;
    const uint32_t st = lds0 + (uint32_t)(n_buf * L::STAGE) + w * 1024;
    const uint64_t kb = (uint64_t)ks * SROW;
#pragma unroll
    for (int i = 0; i < SDMA_P; ++i) dma16(d_poff[i], d_pbase + kb, st + i * (SWAVES * 1024));
#pragma unroll
    for (int i = 0; i < L::DMA_Q; ++i) dma16(d_qoff[i], d_qbase + kb, st + SP_BYTES + i * (SWAVES * 1024));
    n_buf = U(n_buf + 1 == L::NS ? 0 : n_buf + 1);
    if (n_left > 1) {
      --n_left;
      if (++n_ks == ksteps) {
        n_ks = 0;
        ++n_r;
      }
    }
  };

  // ---- fragments --------------------------------------------------------------
  const int r32 = l & 31;
  const int half = l >> 5;
  const int fa = cswz(r32);

  if constexpr (GATHER) {
    load_ids(0);
    wait_vm<0>();
  }
  for (int s = 0; s < L::NS - 1; ++s) issue();

  int buf = 0;
  for (int r = 0; r < nmy; ++r) {
    int qt, pt;
    tile_at(r, qt, pt);
    const int4 ti = sload_int4(a.table + qt);
    const int row0 = ti.y, row1 = ti.z;
    const int nblk = (row1 - row0 + 31) >> 5;  // 32-row token blocks of the tile
    floatx16_t acc[NPB][L::NJ];
#pragma unroll
    for (int p = 0; p < NPB; ++p)
#pragma unroll
      for (int j = 0; j < L::NJ; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[p][j][v] = 0.f;
    for (int ks = 0; ks < ksteps; ++ks) {
      // the oldest stage has landed for every wave, and every wave has read
      // the previous stage, whose buffer the new DMAs go to
      wait_vm_barrier<(L::NS - 2) * L::IPW>();
      issue();
      if (wq < nblk) {
        const char* st = smem + buf * L::STAGE;
        const char* pa = st + (32 * wp + r32) * SROW;
        const char* pb = st + SP_BYTES + (32 * wq + r32) * SROW;
        bf16x8_t fp[NPB][4], fq[L::NJ][4];
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
#pragma unroll
          for (int p = 0; p < NPB; ++p)
            fp[p][kk] = *(const bf16x8_t*)(pa + p * 128 * SROW + (((2 * kk + half) ^ fa ^ (4 * (wp & 1))) << 4));
#pragma unroll
          for (int j = 0; j < L::NJ; ++j)
            fq[j][kk] = *(const bf16x8_t*)(pb + j * 64 * SROW + (((2 * kk + half) ^ fa ^ (4 * wq)) << 4));
        }
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
#pragma unroll
          for (int j = 0; j < L::NJ; ++j)
#pragma unroll
            for (int p = 0; p < NPB; ++p)
              acc[p][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fp[p][kk], fq[j][kk], acc[p][j], 0, 0, 0);
      }
      buf = U(buf + 1 == L::NS ? 0 : buf + 1);
    }

    // ---- epilogue: acc[p][j][4 g + i] is (token row 32 (wq + 2 j) + r32,
    //      tile weight row 32 (wp + 4 p) + 8 g + 4 half + i); H % 64 == 0
    //      and N % 128 == 0 make column validity uniform over a block
#pragma unroll
    for (int j = 0; j < L::NJ; ++j) {
      if (wq + 2 * j >= nblk) continue;
      const int qrow = 32 * (wq + 2 * j) + r32;
      const int gq = row0 + qrow;
      const bool row_ok = gq < row1;
      if constexpr (EPI == EPI_SWIGLU) {
        const float lim = a.limit;
        const bool clamp = lim == lim;
#pragma unroll
        for (int p = 0; p < NPB; ++p) {
          uint32_t gp[2][2], up[2][2], ap[2][2];
#pragma unroll
          for (int g = 0; g < 2; ++g) {
#pragma unroll
            for (int i2 = 0; i2 < 2; ++i2) {
              // h is materialised in bf16 by the reference; SwiGLU reads it
              gp[g][i2] = pack_bf16x2(acc[p][j][8 * g + 2 * i2], acc[p][j][8 * g + 2 * i2 + 1]);
              up[g][i2] = pack_bf16x2(acc[p][j][8 * g + 4 + 2 * i2], acc[p][j][8 * g + 4 + 2 * i2 + 1]);
              float av[2];
#pragma unroll
              for (int h2 = 0; h2 < 2; ++h2) {
                float gc = __uint_as_float(h2 ? (gp[g][i2] & 0xffff0000u) : (gp[g][i2] << 16));
                float uc = __uint_as_float(h2 ? (up[g][i2] & 0xffff0000u) : (up[g][i2] << 16));
                if (clamp) {
                  gc = clamp_max_nan(gc, lim);
                  uc = clamp_nan(uc, lim);
                }
                av[h2] = silu_f(gc) * uc;
              }
              ap[g][i2] = pack_bf16x2(av[0], av[1]);
            }
          }
          // columns 16 (wp + 4 p) + 8 g + 4 half .. + 3 of the tile's STP / 2
          if (row_ok && pt * COLS + 16 * (wp + 4 * p) < a.n_p) {
            const int col = pt * COLS + 16 * (wp + 4 * p) + 4 * half;
            bf16_t* orow = a.out + (int64_t)gq * a.ldo + col;
#pragma unroll
            for (int g = 0; g < 2; ++g) *(uint2*)(orow + 8 * g) = make_uint2(ap[g][0], ap[g][1]);
            if (a.h_out) {
              bf16_t* hrow = a.h_out + (int64_t)gq * a.ldh + col;
#pragma unroll
              for (int g = 0; g < 2; ++g) {
                *(uint2*)(hrow + 8 * g) = make_uint2(gp[g][0], gp[g][1]);
                *(uint2*)(hrow + a.hidden + 8 * g) = make_uint2(up[g][0], up[g][1]);
              }
            }
          }
        }
      } else {
        float sc = 1.f;
        int orow_idx = gq;
        if constexpr (EPI == EPI_SCATTER) {
          const int* meta = (const int*)(smem + L::RING + (r % META_SLOTS) * L::META);
          if (a.dest) orow_idx = min(max(meta[qrow], 0), a.n_dest - 1);
          if (a.row_scale) {
            sc = __int_as_float(meta[TQ + qrow]);
            if (a.scale_sigmoid) sc = sigmoid_f(sc);
          }
        }
        bf16_t* orow = a.out + (int64_t)orow_idx * a.ldo;
#pragma unroll
        for (int p = 0; p < NPB; ++p) {
          uint32_t pk[4][2];
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            pk[g][0] = pack_bf16x2(acc[p][j][4 * g] * sc, acc[p][j][4 * g + 1] * sc);
            pk[g][1] = pack_bf16x2(acc[p][j][4 * g + 2] * sc, acc[p][j][4 * g + 3] * sc);
          }
          // lanes l and l ^ 32 swap one 4-column group each (as in
          // gemm_fwd.hip): every store is 16 bytes
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            uint32_t x[2], y[2];
#pragma unroll
            for (int d = 0; d < 2; ++d) {
              const auto sw = __builtin_amdgcn_permlane32_swap(pk[2 * c][d], pk[2 * c + 1][d], false, false);
              x[d] = sw[0];
              y[d] = sw[1];
            }
            u32x4_t val = u32x4_t{x[0], x[1], y[0], y[1]};
            const int col = pt * COLS + 32 * (wp + 4 * p) + 16 * c + 8 * half;
            if (row_ok && pt * COLS + 32 * (wp + 4 * p) < a.n_p) {
              if (a.accumulate) {
                // add to the row already there (bf16 + bf16, one rounding)
                const u32x4_t prev = *(const u32x4_t*)(orow + col);
#pragma unroll
                for (int d = 0; d < 4; ++d)
                  val[d] = pack_bf16x2(bf16_to_f32(val[d] & 0xffffu) + bf16_to_f32(prev[d] & 0xffffu),
                                       bf16_to_f32(val[d] >> 16) + bf16_to_f32(prev[d] >> 16));
              }
              *(u32x4_t*)(orow + col) = val;
            }
          }
        }
      }
    }
  }
  wait_vm<0>();  // DMAs past the end have landed before the workgroup exits
}

template <int EPI, bool GATHER, int TQ, int STP>
hipError_t launch_tile(FwdArgs a, hipStream_t stream) {
  // set once per process (thread-safe static initialisation)
  static const hipError_t attr_err = hipFuncSetAttribute((const void*)gg_small_kernel<EPI, GATHER, TQ, STP>,
                                                         hipFuncAttributeMaxDynamicSharedMemorySize, Geo<TQ, STP>::LDS);
  if (attr_err != hipSuccess) return attr_err;
  constexpr int COLS = EPI == EPI_SWIGLU ? STP / 2 : STP;
  a.np_tiles = (a.n_p + COLS - 1) / COLS;
  const int grid = (num_cus() + 7) & ~7;
  return launch_k(true, gg_small_kernel<EPI, GATHER, TQ, STP>, dim3(grid), dim3(64 * SWAVES), Geo<TQ, STP>::LDS, stream,
                  a);
}

template <int EPI, bool GATHER>
hipError_t launch_epi(const FwdArgs& a, int rows, int cols, hipStream_t stream) {
  if (rows == 64)
    return cols == 128 ? launch_tile<EPI, GATHER, 64, 128>(a, stream) : launch_tile<EPI, GATHER, 64, 256>(a, stream);
  return cols == 128 ? launch_tile<EPI, GATHER, 128, 128>(a, stream) : launch_tile<EPI, GATHER, 128, 256>(a, stream);
}

}  // namespace

hipError_t launch_small_gemm(int epi, FwdArgs a, int rows, int cols, hipStream_t stream) {
  if (epi == EPI_SWIGLU)
    return a.q_index ? launch_epi<EPI_SWIGLU, true>(a, rows, cols, stream)
                     : launch_epi<EPI_SWIGLU, false>(a, rows, cols, stream);
  if (epi == EPI_SCATTER) return launch_epi<EPI_SCATTER, false>(a, rows, cols, stream);
  return launch_epi<EPI_STORE, false>(a, rows, cols, stream);
}

}  // namespace ttamd
