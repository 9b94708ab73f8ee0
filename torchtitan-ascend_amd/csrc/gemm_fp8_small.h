// fp8 (e4m3) grouped GEMM with 128 x 128 block scales for few rows per expert
// or few tiles on MI355X (gfx950): the small-tile form of gemm_fp8.hip, as
// gemm_small.hip is of gemm_fwd.hip.
//
//   out[q, p] = sum_kb  sx[kb, q] * sw[e(q), p / 128, kb] *
//                       sum_{k in block kb} xq[q, k] * wq[e(q), p, k]
//
// With few rows per expert the path streams the hit experts' weights; the
// 256 x 256 kernel keeps one 66 KB stage in flight and waits for all of it at
// every stage barrier, and with few tiles leaves CUs idle.  Here a ring of NS
// stages (k in stages of 128 = one scale block, 128-byte rows) is refilled
// with counted waits, NS - 2 whole stages staying in flight across every
// barrier.  Tiles of 64 or 128 token rows x 128 or 256 weight rows; per stage
// every wave issues its weight and token rows and one 4-byte DMA of scales
// (waves below TQ / 64 the row scales, the others the weight-block scales of
// the tile's 16-row blocks, the same values from each).
//
// 8 waves as 2 (token) x 4 (weight): wave (wq, wp) owns the 32-row weight
// blocks wp, wp + 4 (two 16-row blocks each; SWIGLU: 16 gate rows and the 16
// matching up rows) and the 16-row token blocks wq, wq + 2, ...; one
// v_mfma_f32_16x16x128_f8f6f4 covers a block's whole scale block and its sum
// goes into the fp32 accumulator times sx * sw, as in gemm_fp8.hip.
//
// Measured (expert stage of a DeepSeek-V3 shard, 32 experts of 7168 x 2048:
// gather + quantise, both GEMMs, one box): 32 rows 320 -> 214 us, 200 rows 370
// -> 281, 1000 rows 385 -> 305, 3000 rows 430 -> 369; w13 at 200 rows 184 ->
// 141 us (5.8 TB/s of weights; its tables and the two quantisations are the
// rest).
#pragma once

#include "common.h"
#include "dma_asm.h"
#include "gemm_common.h"
#include "kernels.h"

namespace ttamd {
namespace fp8_small {

using namespace dma;

constexpr int SKB = 128;  // k per stage: bytes per row
constexpr int SWAVES = 8;
constexpr int META_SLOTS = 8;  // EPI_SCATTER row metadata, tile round % 8

typedef int i32x8_t __attribute__((ext_vector_type(8)));

template <int TQ, int STP>
struct Geo {
  static constexpr int NS = STP == 256 ? 3 : TQ == 64 ? 6 : 4;
  static constexpr int DMA_P = STP / 8 / SWAVES;
  static constexpr int DMA_Q = TQ / 8 / SWAVES;
  static constexpr int IPW = DMA_P + DMA_Q + 1;  // DMAs per wave and stage
  static constexpr int NPB = STP / 64;           // 16-row weight blocks per wave
  static constexpr int NJ = TQ / 32;             // 16-row token blocks per wave
  static constexpr int P_BYTES = STP * SKB;
  static constexpr int SX_OFF = P_BYTES + TQ * SKB;
  static constexpr int SW_OFF = SX_OFF + TQ * 4;
  static constexpr int STAGE = SW_OFF + 256;
  static constexpr int RING = NS * STAGE;
  static constexpr int META = TQ * 8;
  static constexpr int LDS = RING + META_SLOTS * META;
  static_assert(LDS <= 160 * 1024, "LDS of a CU");
};

// One workgroup's share of a GEMM over nqt token tiles of at most TQ rows.
template <int EPI, int TQ, int STP>
__device__ __forceinline__ void run(const Fp8Args& a, const int4* table, int nqt, int np_tiles) {
  using L = Geo<TQ, STP>;
  constexpr int NPB = L::NPB, NJ = L::NJ;
  constexpr int COLS = EPI == EPI_SWIGLU ? STP / 2 : STP;  // output columns per tile
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wq = w >> 2;
  const int wp = w & 3;
  const int l = threadIdx.x & 63;
  const int G = gridDim.x;
  const int b = blockIdx.x;
  auto U = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
  const int ntiles = nqt * np_tiles;
  const int ksteps = U(a.kred / SKB);
  // walk, tile order and k rotation as in gemm_small.hip
  const int R = U(ntiles / G);
  const int rt = ntiles - R * G;
  const int slot = (b & 7) * (G >> 3) + (b >> 3);
  const int nmy = R + (b < rt ? 1 : 0);
  if (nmy == 0) return;
  const int total = nmy * ksteps;
  auto tile_at = [&](int r, int& qt, int& pt) {
    const int t = r < R ? r * G + slot : R * G + b;
    const int blk = t / (2 * np_tiles);
    const int in_blk = t - blk * 2 * np_tiles;
    const int gq = min(2, nqt - 2 * blk);
    pt = in_blk / gq;
    qt = 2 * blk + (in_blk - pt * gq);
  };
  const int n_cols = EPI == EPI_SWIGLU ? (int)a.hidden : a.n_p;  // output columns

  const uint32_t lds0 = lds_addr(smem);
  const int drow = l >> 3;
  const int rr0 = 8 * w + drow;
  const uint32_t lch16 = (uint32_t)(((l & 7) ^ ((drow ^ w) & 7)) * 16);

  // ---- DMA stream -----------------------------------------------------------
  int d_r = -1, d_rot = 0;
  uint64_t d_pbase = 0, d_qbase = 0, d_scbase = 0, d_scstep = 0;
  uint32_t d_poff[L::DMA_P], d_qoff[L::DMA_Q], d_scoff = 0;
  const uint32_t d_sclds = w < TQ / 64 ? (uint32_t)(L::SX_OFF + w * 256) : (uint32_t)L::SW_OFF;
  auto dma_tile = [&](int r) {
    int qt, pt;
    tile_at(r, qt, pt);
    const int4 ti = sload_int4(table + qt);
    const int qmax = ti.z - ti.y - 1;
    const int last = n_cols - 1 - pt * COLS;
#pragma unroll
    for (int i = 0; i < L::DMA_P; ++i) {
      const int rb = SWAVES * i + w;  // 8-row block of the tile; SWIGLU: 16 gate rows, 16 up rows, ...
      const int row = EPI == EPI_SWIGLU ? ((rb >> 1) & 1 ? (int)a.hidden : 0) + min(16 * (rb >> 2) + 8 * (rb & 1) + drow, last)
                                        : min(8 * rb + drow, last);
      d_poff[i] = (uint32_t)row * (uint32_t)a.ldp + lch16;
    }
#pragma unroll
    for (int i = 0; i < L::DMA_Q; ++i) d_qoff[i] = (uint32_t)min(rr0 + 64 * i, qmax) * (uint32_t)a.ldq + lch16;
    d_pbase = (uint64_t)(a.p + (int64_t)ti.x * a.p_estride + (int64_t)pt * COLS * a.ldp);
    d_qbase = (uint64_t)(a.q + (int64_t)ti.y * a.ldq);
    if (w < TQ / 64) {  // row scales of this k block
      d_scbase = (uint64_t)(a.sx + ti.y);
      d_scoff = (uint32_t)min(64 * w + l, qmax) * 4;
      d_scstep = (uint64_t)a.ldsx * 4;
    } else {  // lane m: the weight-block scale of the tile's 16-row block m
      const int m = min(l, STP / 16 - 1);
      const int row = pt * COLS + (EPI == EPI_SWIGLU ? (m & 1 ? (int)a.hidden : 0) + 16 * (m >> 1) : 16 * m);
      d_scbase = (uint64_t)(a.sw + (int64_t)ti.x * a.sw_estride);
      d_scoff = (uint32_t)min(row >> 7, a.n_p / 128 - 1) * (uint32_t)ksteps * 4;
      d_scstep = 4;
    }
    d_rot = a.ldp % 4096 == 0 ? U((5 * pt + 3 * ti.x) % ksteps) : 0;
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
  int n_r = 0, n_ks = 0, n_left = total, n_buf = 0;
  auto issue = [&]() {
    if (n_r != d_r) dma_tile(n_r);
    int ks = n_ks + d_rot;
    ks = ks >= ksteps ? ks - ksteps : ks;
    const uint32_t st = lds0 + (uint32_t)(n_buf * L::STAGE);
    const uint64_t kb = (uint64_t)ks * SKB;
#pragma unroll
    for (int i = 0; i < L::DMA_P; ++i) dma16(d_poff[i], d_pbase + kb, st + w * 1024 + i * (SWAVES * 1024));
#pragma unroll
    for (int i = 0; i < L::DMA_Q; ++i) dma16(d_qoff[i], d_qbase + kb, st + L::P_BYTES + w * 1024 + i * (SWAVES * 1024));
    dma4(d_scoff, d_scbase + (uint64_t)ks * d_scstep, st + d_sclds);
    n_buf = U(n_buf + 1 == L::NS ? 0 : n_buf + 1);
    if (n_left > 1) {
      --n_left;
      if (++n_ks == ksteps) {
        n_ks = 0;
        ++n_r;
      }
    }
  };

  // ---- fragments: lane l holds bytes 32 (l / 16) .. + 31 of row l % 16 ----------
  const int r16 = l & 15;
  const int g4 = l >> 4;
  const int f16 = cswz(r16);
  auto frag16 = [&](const char* base, int m) {  // 16-row block m
    const int x = f16 ^ ((2 * m) & 6);
    const char* row = base + (16 * m + r16) * SKB;
    const i32x4_t lo = *(const i32x4_t*)(row + (((2 * g4) ^ x) * 16));
    const i32x4_t hi = *(const i32x4_t*)(row + (((2 * g4 + 1) ^ x) * 16));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  auto pblk = [&](int pb) { return 2 * (wp + 4 * (pb >> 1)) + (pb & 1); };  // the wave's weight block pb

  for (int s = 0; s < L::NS - 1; ++s) issue();

  int buf = 0;
  for (int r = 0; r < nmy; ++r) {
    int qt, pt;
    tile_at(r, qt, pt);
    const int4 ti = sload_int4(table + qt);
    const int row0 = ti.y, row1 = ti.z;
    const int nblk = (row1 - row0 + 15) >> 4;  // 16-row token blocks of the tile
    floatx4_t acc[NPB][NJ];
#pragma unroll
    for (int p = 0; p < NPB; ++p)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[p][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    for (int ks = 0; ks < ksteps; ++ks) {
      // the oldest stage has landed for every wave, and every wave has read
      // the previous stage, whose buffer the new DMAs go to
      wait_vm_barrier<(L::NS - 2) * L::IPW>();
      issue();
      if (wq < nblk) {
        const char* st = smem + buf * L::STAGE;
        i32x8_t fa[NPB];
        float swv[NPB];
#pragma unroll
        for (int p = 0; p < NPB; ++p) {
          fa[p] = frag16(st, pblk(p));
          swv[p] = *(const float*)(st + L::SW_OFF + pblk(p) * 4);
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          if (wq + 2 * j < nblk) {  // wave-uniform
            const int m = wq + 2 * j;
            const i32x8_t fb = frag16(st + L::P_BYTES, m);
            const float sx = *(const float*)(st + L::SX_OFF + (16 * m + r16) * 4);
#pragma unroll
            for (int p = 0; p < NPB; ++p) {
              const floatx4_t z = {};
              // (zero scale operands: the unscaled v_mfma_f32_16x16x128_f8f6f4)
              const floatx4_t part = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fa[p], fb, z, 0, 0, 0, 0, 0, 0);
              const float sc = swv[p] * sx;
#pragma unroll
              for (int v = 0; v < 4; ++v) acc[p][j][v] += part[v] * sc;
            }
          }
        }
      }
      buf = U(buf + 1 == L::NS ? 0 : buf + 1);
    }

    // ---- epilogue: acc[p][j][i] is (token row 16 (wq + 2 j) + r16, tile
    //      weight row 16 pblk(p) + 4 g4 + i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      if (wq + 2 * j >= nblk) continue;
      const int qrow = 16 * (wq + 2 * j) + r16;
      const int gq = row0 + qrow;
      const bool row_ok = gq < row1;
      if constexpr (EPI == EPI_SWIGLU) {
        const float lim = a.limit;
        const bool clamp = lim == lim;
#pragma unroll
        for (int p = 0; p < NPB; p += 2) {
          const int col = pt * COLS + 16 * (wp + 2 * p);  // 32-row block wp + 4 (p / 2): 16 columns
          float av[4], gv[4], uv[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            gv[i] = round_bf16(acc[p][j][i]);
            uv[i] = round_bf16(acc[p + 1][j][i]);
            float gc = gv[i], uc = uv[i];
            if (clamp) {
              gc = clamp_max_nan(gc, lim);
              uc = clamp_nan(uc, lim);
            }
            av[i] = silu_f(gc) * uc;
          }
          if (row_ok && col < n_cols) {
            bf16_t* orow = a.out + (int64_t)gq * a.ldo + col + 4 * g4;
            *(uint2*)orow = make_uint2(pack_bf16x2(av[0], av[1]), pack_bf16x2(av[2], av[3]));
            if (a.h_out) {
              bf16_t* hrow = a.h_out + (int64_t)gq * a.ldh + col + 4 * g4;
              *(uint2*)hrow = make_uint2(pack_bf16x2(gv[0], gv[1]), pack_bf16x2(gv[2], gv[3]));
              *(uint2*)(hrow + a.hidden) = make_uint2(pack_bf16x2(uv[0], uv[1]), pack_bf16x2(uv[2], uv[3]));
            }
          }
        }
      } else {
        float scl = 1.f;
        int orow_idx = gq;
        if constexpr (EPI == EPI_SCATTER) {
          const int* meta = (const int*)(smem + L::RING + (r % META_SLOTS) * L::META);
          if (a.dest) orow_idx = min(max(meta[qrow], 0), a.n_dest - 1);
          if (a.row_scale) scl = __int_as_float(meta[TQ + qrow]);
        }
        bf16_t* orow = a.out + (int64_t)orow_idx * a.ldo;
#pragma unroll
        for (int p = 0; p < NPB; ++p) {
          const int col = pt * COLS + 16 * pblk(p);
          const floatx4_t& v = acc[p][j];
          if (row_ok && col < n_cols)
            *(uint2*)(orow + col + 4 * g4) = make_uint2(pack_bf16x2(v[0] * scl, v[1] * scl), pack_bf16x2(v[2] * scl, v[3] * scl));
        }
      }
    }
  }
  wait_vm<0>();  // DMAs past the end have landed before the workgroup exits
}

}  // namespace fp8_small
}  // namespace ttamd
