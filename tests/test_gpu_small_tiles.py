"""GPU parity of the grouped GEMMs on each of their tilings.

The small tiles (few rows per expert, few tiles): cases at the edges of their
choices, 64- and 128-row tiles, 128 and 256 weight rows (the last tile half
full), one row, a full tile and one row more, empty experts, k of one stage
and of fewer stages than the ring, and rows a multiple of 4 KB apart (the k
walk then starts elsewhere per tile).  The large ones (320 x 256, in fp8 256
x 256): every token-block count, weight rows that leave the last tile part
full, few k stages, the clamp and the saved pre-activation.  Each case names
the tile it is meant for, asserted from the library's own choice.

Tolerance: the inputs are bf16 and the sums fp32, so an output is off by
its bf16 rounding (2^-9 relative, and the pre-activation's once more through
the SwiGLU); 1e-2 of the row's largest value covers both.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from gpu_util import DEV, announce, assert_close, bf16_dev, f32_dev, rand_bf16, to_np
from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu
TOL = 1e-2

# rows per expert, N (or H for the SwiGLU: 2 H weight rows), K, and the tile
# of the store / scatter (N) and of the SwiGLU (2 H) GEMM
CASES = [
    ((1,), 128, 64, (64, 128), (64, 128)),                        # one row, one k stage
    ((0, 1, 0, 2, 1), 192, 2048, (64, 128), (64, 128)),           # rotated k walk
    ((64, 65, 33, 1, 0, 63), 320, 192, (64, 128), (64, 128)),     # 64-row tiles and one row past
    ((5,) * 300, 384, 320, (64, 128), (64, 256)),                 # more than one round, fewer stages than the ring
    ((9,) * 200 + (0,) * 20 + (64,) * 3, 1664, 256, (64, 256), (64, 256)),  # last 256-row tile of N half full
    ((9,) * 200 + (0,) * 20 + (64,) * 3, 448, 256, (64, 256), (64, 256)),   # ... and of H (H % 128 == 64)
    ((128, 129, 97, 1, 300, 0, 31, 128, 90), 448, 384, (128, 128), (128, 128)),  # 128-row tiles and one row past
    ((90, 100, 128, 70, 96) * 26, 1152, 2048, (128, 256), (128, 256)),  # whole and partial rounds, rotated, N half full
    ((128, 129, 97, 1, 300, 0, 31) * 2, 1216, 256, (128, 128), (128, 256)),  # H % 128 == 64
    ((700, 1300), 640, 1024, (128, 128), (128, 128)),             # more rows per expert, too few tiles for the large kernel
]

# every 32-row token block count, one row past a tile, tall experts in several
# tiles of near-equal height, empty ones; twice, so that the row count is past
# the small tiles' range
HEIGHTS = (1, 31, 32, 33, 64, 65, 96, 97, 128, 129, 160, 161, 192, 193, 224, 256, 257, 288, 289, 319, 320, 321, 0, 640, 700) * 2
LARGE = (320, 256)
LARGE_CASES = [
    (HEIGHTS, 192, 64, LARGE, LARGE),                             # one k stage; H % 128 == 64
    (HEIGHTS[::-1], 320, 128, LARGE, LARGE),                      # two stages; last tile of H and of N half full
    (HEIGHTS, 640, 192, LARGE, LARGE),                            # three stages; N half full
    ((8200, 0, 100), 448, 2048, LARGE, LARGE),                    # 26 tiles of one expert, rotated k walk
]


ALL_CASES = CASES + LARGE_CASES


def _case(i):
    counts, n, k, tile_n, tile_2h = ALL_CASES[i]
    counts = np.array(counts, np.int64)
    rng = np.random.default_rng(100 + i)
    return counts, int(counts.sum()), len(counts), n, k, rng, tile_n, tile_2h


def _offs(counts):
    return torch.from_numpy(np.cumsum(counts).astype(np.int32)).to(DEV)


@pytest.mark.parametrize("i", range(len(ALL_CASES)))
@pytest.mark.parametrize("limit", [None, 0.5])
def test_small_swiglu(ops, i, limit):
    counts, M, E, H, D, rng, _, tile = _case(i)
    assert ops.gemm_tiles(counts, 2 * H, D)[:2] == tile
    T = (M + 1) // 2
    tok, w13 = rand_bf16(rng, (T, D)), rand_bf16(rng, (E, 2 * H, D), 0.05)
    src = rng.integers(0, 2 * T, M).astype(np.int32)
    announce(f"small swiglu M={M} E={E} H={H} D={D} limit={limit}")
    wd, od = bf16_dev(w13), _offs(counts)
    h_ref = O.bf16_round(O.grouped_mm(tok[src // 2], w13, np.cumsum(counts)))
    a_ref = O.swiglu(h_ref, limit)
    a, h = ops.grouped_mm_swiglu(bf16_dev(tok[src // 2]), wd, od, limit, save_h=True)
    assert_close(to_np(h), h_ref, TOL, "h")
    assert_close(to_np(a), a_ref, 2 * TOL, "a")
    if D >= 128:
        a2, h2 = ops.grouped_mm_swiglu_gather(bf16_dev(tok), torch.from_numpy(src).to(DEV), 2, wd, od, limit, save_h=True)
        assert torch.equal(a, a2) and torch.equal(h, h2), "gathered rows differ from the same rows given in order"


@pytest.mark.parametrize("i", range(len(ALL_CASES)))
def test_small_store_and_scatter(ops, i):
    counts, M, E, N, K, rng, tile, _ = _case(i)
    N = -(-N // 128) * 128
    assert ops.gemm_tiles(counts, N, K)[:2] == tile
    x, w = rand_bf16(rng, (M, K)), rand_bf16(rng, (E, N, K), 0.05)
    dest = rng.permutation(M).astype(np.int32)
    scale = rng.random(M).astype(np.float32)
    announce(f"small store / scatter M={M} E={E} N={N} K={K}")
    xd, wd, od = bf16_dev(x), bf16_dev(w), _offs(counts)
    y = O.grouped_mm(x, w, np.cumsum(counts))
    assert_close(to_np(ops.grouped_mm(xd, wd, od)), y, TOL, "store")
    out = ops.grouped_mm_unpermute(xd, wd, od, f32_dev(scale), torch.from_numpy(dest).to(DEV), M)
    ref = np.zeros((M, N), np.float32)
    ref[dest] = y * scale[:, None]
    assert_close(to_np(out), ref, TOL, "scatter")


@pytest.mark.parametrize("T,D,H,tile_rows", [(1, 128, 64, 64), (70, 256, 192, 64), (900, 512, 448, 128),
                                             (8300, 384, 192, 320)])
def test_small_shared_expert(ops, T, D, H, tile_rows):
    """The accumulating, gated epilogue (one expert with every row)."""
    assert ops.gemm_tiles((T,), D, H)[0] == tile_rows
    rng = np.random.default_rng(T)
    x, w13, w2 = rand_bf16(rng, (T, D)), rand_bf16(rng, (1, 2 * H, D), 0.05), rand_bf16(rng, (1, D, H), 0.05)
    base, gate = rand_bf16(rng, (T, D)), rng.standard_normal(T).astype(np.float32)
    announce(f"small shared expert T={T} D={D} H={H}")
    out = ops.shared_expert_add(bf16_dev(base), bf16_dev(x), bf16_dev(w13[0]), bf16_dev(w2[0]), f32_dev(gate))
    a = O.bf16_round(O.swiglu(O.bf16_round(O.grouped_mm(x, w13, np.array([T])))))
    y = O.bf16_round(O.grouped_mm(a, w2, np.array([T])) / (1 + np.exp(-gate[:, None])))
    assert_close(to_np(out), base + y, TOL, "out")


# The same of the fp8 form: K a multiple of 128
FP8_CASES = [
    ((1,), 128, 128, (64, 128), (64, 128)),                       # one row, one k stage
    ((0, 1, 0, 2, 1), 192, 4096, (64, 128), (64, 128)),           # up rows straddle scale blocks, rotated k walk
    ((64, 65, 33, 1, 0, 17, 16, 63), 320, 384, (64, 128), (64, 128)),  # 64-row tiles and one row past, 16-row block edges
    ((9,) * 200 + (0,) * 20 + (64,) * 3, 1152, 256, (64, 256), (64, 256)),  # last 256-row tile of N half full
    ((9,) * 200 + (0,) * 20 + (64,) * 3, 448, 256, (64, 256), (64, 256)),   # ... and of H (H % 128 == 64)
    ((128, 129, 97, 1, 300, 0, 31, 128, 90), 448, 640, (128, 128), (128, 128)),  # 128-row tiles and one row past
    ((90, 100, 128, 70, 96) * 26, 1152, 512, (128, 128), (128, 256)),  # whole and partial rounds
]


# The same of the 256 x 256 fp8 tiles: every 16-row block count in both halves,
# walks of 1 to 4 tiles per workgroup, with 1 to 3 k stages of 128
FP8_HEIGHTS = (1, 16, 17, 40, 64, 97, 128, 129, 144, 161, 200, 230, 256, 257, 300, 512)
FP8_LARGE = (256, 256)
FP8_LARGE_CASES = [
    (FP8_HEIGHTS * 4, 3072, 128, FP8_LARGE, FP8_LARGE),
    (FP8_HEIGHTS * 4, 1152, 256, FP8_LARGE, FP8_LARGE),
    (FP8_HEIGHTS[::-1] * 4, 1024, 384, FP8_LARGE, FP8_LARGE),
    (FP8_HEIGHTS * 4, 320, 256, FP8_LARGE, FP8_LARGE),            # H % 128 == 64: up rows straddle scale blocks
]


@pytest.mark.parametrize("i", range(len(FP8_CASES)))
def test_small_fp8(ops, i):
    """Every epilogue of the fp8 small tiles against the dequantising oracle
    (operands e4m3 with fp32 block scales, so only the sums' fp32 rounding
    and the output's bf16 rounding differ)."""
    _check_fp8(ops, *FP8_CASES[i], 200 + i)


@pytest.mark.parametrize("i", range(len(FP8_LARGE_CASES)))
def test_large_fp8_stage_pipeline(ops, i):
    """The same for the large fp8 tiles, whose fragment reads, scale FMAs and
    DMAs run across the stage and tile boundaries."""
    _check_fp8(ops, *FP8_LARGE_CASES[i], 300 + i)


def _check_fp8(ops, counts, n, K, tile_n, tile_2h, seed):
    counts = np.array(counts, np.int64)
    M, E = int(counts.sum()), len(counts)
    offs_h, od = np.cumsum(counts), _offs(counts)
    rng = np.random.default_rng(seed)
    H, N = -(-n // 64) * 64, -(-n // 128) * 128
    assert (ops.gemm_tiles(counts, N, K, True)[:2], ops.gemm_tiles(counts, 2 * H, K, True)[:2]) == (tile_n, tile_2h)
    x = bf16_dev(rand_bf16(rng, (M, K)))
    announce(f"fp8 tiles M={M} E={E} n={n} K={K}")
    xq, sx = ops.quantize_fp8_rows(x)
    xd = O.e4m3_bits_to_f32(xq.cpu().numpy()).reshape(M, K // 128, 128) * sx.cpu().numpy().T[:, :, None]
    xd = xd.reshape(M, K)

    def weights(rows):
        w = bf16_dev(rand_bf16(rng, (E, rows, K), 0.05))
        q, s = ops.quantize_fp8_blocks(w)
        d = O.e4m3_bits_to_f32(q.cpu().numpy()).reshape(E, rows // 128, 128, K // 128, 128)
        return q, s, (d * s.cpu().numpy()[:, :, None, :, None]).reshape(E, rows, K)

    wq, sw, wd = weights(N)
    y = O.grouped_mm(xd, wd, offs_h)
    assert_close(to_np(ops.grouped_mm_fp8(xq, sx, wq, sw, od)), y, TOL, "store")
    dest, scale = rng.permutation(M).astype(np.int32), rng.random(M).astype(np.float32)
    out = ops.grouped_mm_fp8_unpermute(xq, sx, wq, sw, od, f32_dev(scale), torch.from_numpy(dest).to(DEV), M)
    ref = np.zeros((M, N), np.float32)
    ref[dest] = y * scale[:, None]
    assert_close(to_np(out), ref, TOL, "scatter")
    wq, sw, wd = weights(2 * H)
    h_ref = O.bf16_round(O.grouped_mm(xd, wd, offs_h))
    for limit in (None, 0.5):
        a, h = ops.grouped_mm_fp8_swiglu(xq, sx, wq, sw, od, limit, save_h=True)
        assert_close(to_np(h), h_ref, TOL, "h")
        assert_close(to_np(a), O.swiglu(h_ref, limit), 2 * TOL, "a")


# rows per expert, N (or H), K of calls whose tile counts decide between the
# 128-row and the 256-row tiles on the device, with the tile expected of the
# store / scatter (N) and the SwiGLU (2 H) GEMM: both sides and both widths of
# the small one, the same row total even and on few experts
FP8_PICK_CASES = [
    ((107,) * 24, 1920, 512, (128, 256), (128, 256)),
    ((130,) * 10 + (90,) * 14, 1920, 384, (256, 256), (128, 256)),  # the same rows near enough: one more small round
    ((97,) * 14, 1152, 384, (128, 128), (128, 256)),
    ((120,) * 60, 640, 256, (128, 256), (128, 128)),
    ((900,) * 8, 2048, 512, (256, 256), (256, 256)),
    ((7000, 1, 129, 0, 33, 0, 0, 255), 1088, 256, (128, 128), (256, 256)),  # up rows straddle scale blocks
]


@pytest.mark.parametrize("i", range(len(FP8_PICK_CASES)))
def test_fp8_tiles_chosen_by_the_plan(ops, i):
    _check_fp8(ops, *FP8_PICK_CASES[i], 400 + i)


@pytest.mark.parametrize("R", [1, 4, 5, 8191, 8193])
def test_fp8_row_quantiser_row_groups(ops, R):
    """Few rows run one per wave, many four per wave: the same codes and
    scales either way (the rows of a larger call)."""
    rng = np.random.default_rng(R)
    K = 256
    x = bf16_dev(rand_bf16(rng, (R, K)))
    big = torch.cat([x, bf16_dev(rand_bf16(rng, (20000, K)))])
    announce(f"fp8 row quantiser R={R}")
    q, s = ops.quantize_fp8_rows(x)
    q2, s2 = ops.quantize_fp8_rows(big)
    assert torch.equal(q, q2[:R]) and torch.equal(s, s2[:, :R])


def test_large_tiles_split_epilogues_and_replay(ops):
    """35 experts of 320 rows keep the 320 x 256 kernel, whose 24 leftover
    tiles (of 280) are cut along k: the SwiGLU epilogue (with and without the
    gather) and the scatter one, and replays of the captured pair with other
    work in between (the plan's arrival counters must return to zero)."""
    E, D, H = 35, 2048, 1024
    counts = np.full(E, 320)
    M = int(counts.sum())
    rng = np.random.default_rng(7)
    labels = rng.permutation(np.repeat(np.arange(E), counts))
    sidx = O.stable_order(labels, E).astype(np.int32)
    x, w13 = rand_bf16(rng, (M, D)), rand_bf16(rng, (E, 2 * H, D), 0.05)
    a, w2 = rand_bf16(rng, (M, 2048)), rand_bf16(rng, (E, D, 2048), 0.05)
    scale = rng.random(M).astype(np.float32)
    announce("large tiles, split swiglu gather / scatter, replayed")
    xd, sd, od, ad, wd13, wd2 = (bf16_dev(x), torch.from_numpy(sidx).to(DEV), _offs(counts), bf16_dev(a),
                                 bf16_dev(w13), bf16_dev(w2))

    def step():
        act, _ = ops.grouped_mm_swiglu_gather(xd, sd, 1, wd13, od)
        return act, ops.grouped_mm_unpermute(ad, wd2, od, f32_dev_scale, sd, M)

    f32_dev_scale = f32_dev(scale)
    act, out = step()
    plain, _ = ops.grouped_mm_swiglu(bf16_dev(x[sidx]), wd13, od)
    assert torch.equal(act, plain)
    h_ref = O.bf16_round(O.grouped_mm(x[sidx], w13, np.cumsum(counts)))
    assert_close(to_np(act), O.swiglu(h_ref), 2 * TOL, "a")
    ref = np.zeros((M, D), np.float32)
    ref[sidx] = O.grouped_mm(a, w2, np.cumsum(counts)) * scale[:, None]
    assert_close(to_np(out), ref, TOL, "out")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        g_act, g_out = step()
    for _ in range(3):
        g_act.zero_(), g_out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(g_act, act) and torch.equal(g_out, out)
        step()
