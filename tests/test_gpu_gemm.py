"""GPU parity of the grouped GEMM kernels against the CPU oracle (fp32
accumulation).  Tolerance: max relative error (max|got-ref| / max|ref|)
<= 2e-2 for bf16, the bound the path is specified to."""
from __future__ import annotations

import importlib

import numpy as np
import pytest
import torch

from gpu_util import DEV, announce, assert_close, bf16_dev, f32_dev, rand_bf16, to_np, zipf_counts
from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu
TOL = 2e-2


def _counts(kind, M, E, rng):
    if kind == "uniform":
        c = np.full(E, M // E)
        c[: M - c.sum()] += 1
        return c
    if kind == "random":
        cut = np.sort(rng.integers(0, M + 1, E - 1))
        return np.diff(np.concatenate([[0], cut, [M]]))
    if kind == "zipf":
        # at least one empty expert whenever E > 1 (E // 8 of them for E >= 16)
        return zipf_counts(M, E, 1.2, max(1, E - max(1, E // 8)), rng)
    if kind == "one":
        c = np.zeros(E, np.int64)
        c[E // 2] = M
        return c
    raise ValueError(kind)


def _offs(counts):
    return torch.from_numpy(np.cumsum(counts).astype(np.int32)).to(DEV)


def _gmm_ref(x, w, counts):
    return O.grouped_mm(x, w, np.cumsum(counts))


CASES = [
    # M, E, N, K, kind
    (1000, 8, 256, 256, "random"),
    (700, 4, 512, 2048, "zipf"),
    (129, 3, 128, 64, "random"),
    (4096, 16, 384, 512, "one"),
    (333, 32, 128, 128, "zipf"),
]


@pytest.mark.parametrize("M,E,N,K,kind", CASES)
def test_grouped_mm(ops, M, E, N, K, kind):
    rng = np.random.default_rng(M + E + N + K)
    counts = _counts(kind, M, E, rng)
    x = rand_bf16(rng, (M, K))
    w = rand_bf16(rng, (E, N, K), 0.05)
    announce(f"grouped_mm M={M} E={E} N={N} K={K} {kind}")
    out = ops.grouped_mm(bf16_dev(x), bf16_dev(w), _offs(counts))
    ref = _gmm_ref(x, w, counts)
    assert_close(to_np(out), ref, TOL, "to_np(out)")


def test_grouped_mm_ignores_rows_past_last_offset(ops):
    rng = np.random.default_rng(1)
    M, E, N, K = 512, 4, 128, 128
    counts = np.array([100, 0, 200, 50])  # 350 of 512 rows grouped
    x = rand_bf16(rng, (M, K))
    w = rand_bf16(rng, (E, N, K), 0.05)
    announce("grouped_mm tail rows")
    out = torch.full((M, N), 7.0, dtype=torch.bfloat16, device=DEV)
    res = ops.grouped_mm(bf16_dev(x), bf16_dev(w), _offs(counts))
    out[:350] = res[:350]
    assert_close(to_np(res)[:350], _gmm_ref(x, w, counts)[:350], TOL, "to_np(res)[:350]")


@pytest.mark.parametrize("limit", [None, 0.75])
@pytest.mark.parametrize("M,E,D,H,kind", [(1000, 8, 256, 128, "random"), (2048, 16, 512, 192, "zipf"),
                                          (96, 2, 128, 64, "one")])
def test_grouped_mm_swiglu(ops, M, E, D, H, kind, limit):
    rng = np.random.default_rng(M + D + H)
    counts = _counts(kind, M, E, rng)
    x = rand_bf16(rng, (M, D))
    w13 = rand_bf16(rng, (E, 2 * H, D), 0.08)
    announce(f"swiglu M={M} E={E} D={D} H={H} {kind} limit={limit}")
    a, h = ops.grouped_mm_swiglu(bf16_dev(x), bf16_dev(w13), _offs(counts), limit, save_h=True)
    h_ref = O.bf16_round(_gmm_ref(x, w13, counts))
    a_ref = O.swiglu(h_ref, limit)
    assert_close(to_np(h), h_ref, TOL, "to_np(h)")
    assert_close(to_np(a), a_ref, TOL, "to_np(a)")
    # the activation is computed from the bf16 pre-activation the kernel stored
    assert_close(to_np(a), O.swiglu(to_np(h), limit), 1e-2, "to_np(a)")


@pytest.mark.parametrize("counts,H", [((400, 100), 2304), ((400, 0, 100, 333), 2304), ((50,), 2304),
                                      ((8200, 320), 2304), ((8300, 0, 100, 1), 2304)])
def test_grouped_mm_swiglu_paired_walk_odd_tiles(ops, counts, H):
    """The SwiGLU kernels walk the token tiles in pairs (weight tile major
    inside a pair); with an odd token-tile count the last pair has one tile,
    and with H / 128 = 18 weight tiles a pair spans more than one XCD's 32
    slots (small tiles up to 8192 rows here, the 320 x 256 ones above).  Every tile must still be computed exactly once: compared in
    full with the oracle, per row."""
    rng = np.random.default_rng(sum(counts) + H)
    counts = np.array(counts, np.int64)
    M, E, D = int(counts.sum()), len(counts), 256
    x = rand_bf16(rng, (M, D))
    w13 = rand_bf16(rng, (E, 2 * H, D), 0.08)
    announce(f"swiglu paired walk counts={tuple(counts)} H={H}")
    assert (ops.gemm_tiles(counts, 2 * H, D)[0] == 320) == (M > 8192)
    a, h = ops.grouped_mm_swiglu(bf16_dev(x), bf16_dev(w13), _offs(counts), None, save_h=True)
    h_ref = O.bf16_round(_gmm_ref(x, w13, counts))
    assert_close(to_np(h), h_ref, TOL, "h")
    assert_close(to_np(a), O.swiglu(h_ref), TOL, "a")


@pytest.mark.parametrize("T,K,E,D,H,kind", [(500, 2, 8, 256, 128, "random"), (1024, 4, 16, 512, 192, "zipf"),
                                            (3000, 1, 4, 2048, 768, "random"), (64, 8, 32, 128, 64, "zipf")])
def test_grouped_mm_swiglu_gather(ops, T, K, E, D, H, kind):
    """The permute gather fused into the w13 loads: routed row j is
    x[sorted_indices[j] // K]; compared with the gathered-then-GEMM oracle."""
    rng = np.random.default_rng(T + K + D)
    M = T * K
    counts = _counts(kind, M, E, rng)
    labels = rng.permutation(np.repeat(np.arange(E), counts))
    sidx = O.stable_order(labels, E).astype(np.int32)
    x = rand_bf16(rng, (T, D))
    w13 = rand_bf16(rng, (E, 2 * H, D), 0.08)
    announce(f"swiglu_gather T={T} K={K} E={E} D={D} H={H} {kind}")
    a, h = ops.grouped_mm_swiglu_gather(bf16_dev(x), torch.from_numpy(sidx).to(DEV), K, bf16_dev(w13),
                                        _offs(counts), None, save_h=True)
    h_ref = O.bf16_round(_gmm_ref(x[sidx // K], w13, counts))
    assert_close(to_np(h), h_ref, TOL, "to_np(h)")
    assert_close(to_np(a), O.swiglu(h_ref), TOL, "to_np(a)")


@pytest.mark.parametrize("topk", [1, 4])
def test_grouped_mm_unpermute_scatter_scale(ops, topk):
    rng = np.random.default_rng(topk)
    T, E, D, H = 300, 8, 256, 128
    M = T * topk
    counts = _counts("random", M, E, rng)
    a = rand_bf16(rng, (M, H))
    w2 = rand_bf16(rng, (E, D, H), 0.08)
    dest = rng.permutation(M).astype(np.int32)
    scale = rng.random(M).astype(np.float32)
    announce(f"unpermute scatter topk={topk}")
    out = ops.grouped_mm_unpermute(bf16_dev(a), bf16_dev(w2), _offs(counts), f32_dev(scale),
                                   torch.from_numpy(dest).to(DEV), M)
    y = _gmm_ref(a, w2, counts) * scale[:, None]
    ref = np.zeros_like(y)
    ref[dest] = y
    assert_close(to_np(out), ref, TOL, "to_np(out)")
    if topk > 1:
        summed = ops.sum_topk(out, topk)
        assert_close(to_np(summed), ref.reshape(T, topk, D).sum(1), TOL, "to_np(summed)")


@pytest.mark.parametrize("M,E,N,K,kind", [(1000, 8, 256, 256, "random"), (700, 4, 1536, 2048, "zipf"),
                                          (200, 5, 64, 384, "random")])
def test_grouped_mm_dgrad(ops, M, E, N, K, kind):
    rng = np.random.default_rng(M * 3 + N)
    counts = _counts(kind, M, E, rng)
    dy = rand_bf16(rng, (M, N))
    w = rand_bf16(rng, (E, N, K), 0.05)
    announce(f"dgrad M={M} E={E} N={N} K={K}")
    dx = ops.grouped_mm_dgrad(bf16_dev(dy), bf16_dev(w), _offs(counts))
    offs = np.cumsum(counts)
    ref = np.zeros((M, K), np.float32)
    s = 0
    for e, t in enumerate(offs):
        ref[s:t] = dy[s:t] @ w[e]
        s = t
    assert_close(to_np(dx), ref, TOL, "to_np(dx)")


@pytest.mark.parametrize("limit", [None, 0.5])
def test_grouped_mm_dgrad_swiglu(ops, limit):
    rng = np.random.default_rng(77)
    M, E, D, H = 900, 6, 256, 256
    counts = _counts("random", M, E, rng)
    dy = rand_bf16(rng, (M, D))
    w2 = rand_bf16(rng, (E, D, H), 0.08)
    h = rand_bf16(rng, (M, 2 * H))
    announce(f"dgrad_swiglu limit={limit}")
    dh, a = ops.grouped_mm_dgrad_swiglu(bf16_dev(dy), bf16_dev(w2), bf16_dev(h), _offs(counts), limit, want_a=True)
    offs = np.cumsum(counts)
    g = np.zeros((M, H), np.float32)
    s = 0
    for e, t in enumerate(offs):
        g[s:t] = dy[s:t] @ w2[e]
        s = t
    gate, up = h[:, :H], h[:, H:]
    mg = np.ones_like(gate)
    mu = np.ones_like(up)
    gc, uc = gate, up
    if limit is not None:
        mg = (gate <= limit).astype(np.float32)
        mu = ((up >= -limit) & (up <= limit)).astype(np.float32)
        gc, uc = np.minimum(gate, limit), np.clip(up, -limit, limit)
    sig = 1 / (1 + np.exp(-gc.astype(np.float64)))
    ref = np.concatenate([g * uc * sig * (1 + gc * (1 - sig)) * mg, g * gc * sig * mu], axis=1)
    got = to_np(dh)
    n = int(offs[-1])
    assert_close(got[:n, :H], ref[:n, :H], TOL, "got[:n, :H]")
    assert_close(got[:n, H:], ref[:n, H:], TOL, "got[:n, H:]")
    assert_close(to_np(a)[:n], O.swiglu(h, limit)[:n], 1e-2, "to_np(a)[:n]")


WGRAD_CASES = [
    # M, E, N, K, kind: one tile, then several 256-wide n and k tiles, ragged
    # at both edges (N = 640 = 2.5 tiles, K = 384 = 1.5 tiles), Zipf loads
    # with empty experts, and one C3 expert slab (N = 2 H rows of w13 at
    # D = 5120: 64 x 20 tiles per expert)
    (1000, 8, 256, 128, "random"),
    (3000, 32, 128, 256, "zipf"),
    (64, 4, 128, 128, "one"),
    (2000, 6, 640, 384, "zipf"),
    (1500, 5, 1536, 2048, "random"),
    (3000, 16, 1152, 640, "zipf"),
    (1100, 2, 16384, 5120, "random"),
]


_WGRAD_REF: dict = {}


def _wgrad_case(M, E, N, K, kind):
    """Inputs and oracle of a wgrad case, computed once for both output
    dtypes (the C3-sized slab's oracle is the expensive part)."""
    key = (M, E, N, K, kind)
    if key not in _WGRAD_REF:
        rng = np.random.default_rng(M + E * 5 + N)
        counts = _counts(kind, M, E, rng)
        dy = rand_bf16(rng, (M, N))
        x = rand_bf16(rng, (M, K))
        _WGRAD_REF.clear()
        _WGRAD_REF[key] = (counts, dy, x, O.grouped_wgrad(dy, x, np.cumsum(counts), E))
    return _WGRAD_REF[key]


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,E,N,K,kind", WGRAD_CASES)
def test_grouped_mm_wgrad(ops, M, E, N, K, kind, out_dtype):
    """dW[e] = dy_e^T x_e, checked norm-wise and per expert slice (an error
    confined to a lightly loaded expert is not hidden by the largest).  The
    C3-sized slab (two experts of dW13 at D = 5120, H = 8192: 64 x 20 tiles
    each) runs with fp32 output (the gradient of fp32 master weights) as
    well as bf16."""
    from gpu_util import assert_close

    counts, dy, x, ref = _wgrad_case(M, E, N, K, kind)
    if kind == "zipf":
        assert (counts == 0).any()
    announce(f"wgrad M={M} E={E} N={N} K={K} {kind} {out_dtype}")
    dw = ops.grouped_mm_wgrad(bf16_dev(dy), bf16_dev(x), _offs(counts), E, out_dtype)
    got = to_np(dw)
    del dw
    for e in np.where(counts == 0)[0]:  # empty experts get exact zeros
        assert not np.any(got[e]), f"expert {e} has no rows but a nonzero gradient"
    tol = 1e-5 if out_dtype == torch.float32 and M < 128 else TOL
    assert_close(got, ref, tol, f"wgrad {kind} N={N} K={K}")


def test_grouped_mm_wgrad_empty_expert_next_to_inf(ops):
    """An expert without rows reads the previous expert's last row as its
    (clamped, masked) stage: an Inf / NaN there must not leak into the empty
    expert's exact-zero gradient."""
    rng = np.random.default_rng(31)
    E, N, K = 4, 256, 384
    counts = np.array([70, 0, 130, 0])
    M = int(counts.sum())
    dy = rand_bf16(rng, (M, N))
    x = rand_bf16(rng, (M, K))
    dy[69, 5] = np.inf  # last row of expert 0, next to empty expert 1
    x[69, 7] = np.nan
    dy[M - 1, 0] = -np.inf  # last row of expert 2, next to empty expert 3
    announce("wgrad empty expert next to inf")
    for out_dtype in (torch.float32, torch.bfloat16):
        got = to_np(ops.grouped_mm_wgrad(bf16_dev(dy), bf16_dev(x), _offs(counts), E, out_dtype))
        assert not np.any(got[1]) and not np.any(got[3]), "Inf/NaN of a neighbouring expert leaked"
        assert np.isfinite(got[2][1:]).all()  # only row n = 0 of expert 2 meets its -Inf


def test_grouped_mm_full_size_linearity_and_samples(ops):
    """Qwen3-30B-A3B w13 at full size (M=65536, E=128, N=1536, K=2048):
    scaling x by 2 scales the output exactly, and sampled rows match the oracle."""
    rng = np.random.default_rng(2)
    M, E, N, K = 65536, 128, 1536, 2048
    counts = _counts("uniform", M, E, rng)
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    w = (torch.randn(E, N, K, device=DEV) * 0.02).to(torch.bfloat16)
    offs = _offs(counts)
    announce("grouped_mm full size")
    out = ops.grouped_mm(x, w, offs)
    out2 = ops.grouped_mm(x * 2, w, offs)
    assert torch.equal(out2, out * 2)
    rows = np.sort(rng.choice(M, 64, replace=False))
    e_of = np.searchsorted(np.cumsum(counts), rows, side="right")
    xs = to_np(x[torch.from_numpy(rows).to(DEV)])
    ref = np.stack([xs[i] @ to_np(w[int(e)]).T for i, e in enumerate(e_of)])
    assert_close(to_np(out[torch.from_numpy(rows).to(DEV)]), ref, TOL, "to_np(out[torch.from_numpy(rows).to(DEV)])")


@pytest.mark.parametrize("M,E,kind", [(20000, 32, "zipf"), (65536, 128, "random"), (3000, 8, "one"), (65536, 128, "uniform")])
def test_tile_table_covers_every_row_once(ops, M, E, kind):
    """The token-tile table the GEMM walks (workspace: int count, then one
    int4 {expert, first row, end row, 0} per tile from byte 16): every row
    in exactly one tile of its expert, an expert's c rows in ceil(c/320)
    tiles of one height (a multiple of 32, the last tile shorter), tiles in
    expert then row order; entries past the count marked -1."""
    rng = np.random.default_rng(M + E)
    counts = _counts(kind, M, E, rng)
    if kind == "random":  # near-uniform around M/E, as top-8 routing gives
        counts = rng.multinomial(M, np.full(E, 1.0 / E))
    offs = _offs(counts)
    N, K = 128, 64
    x, w = bf16_dev(rand_bf16(rng, (M, K))), bf16_dev(rand_bf16(rng, (E, N, K), 0.05))
    lib = ops._lib.load()
    wsb = int(lib.ttamd_gemm_workspace_bytes(M, E))
    ws = torch.full((wsb,), 0x7F, dtype=torch.uint8, device=DEV)
    out = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    announce(f"tile table M={M} E={E} {kind}")
    ops._lib.call("ttamd_grouped_mm", ops._p(x), ops._p(w), ops._p(offs), M, E, N, K, ops._p(out), ops._p(ws), wsb,
                  ops._stream(DEV))
    torch.cuda.synchronize()
    raw = ws.cpu().numpy()
    count = int(raw[:4].view(np.int32)[0])
    max_tiles = M // 128 + E + 1
    split_tiles = 512  # split-tile arrival counters between the header and the table
    assert not raw[16 : 16 + 4 * split_tiles].any(), "split-tile counters must be back at zero"
    tab_off = 16 + 4 * split_tiles
    tab = raw[tab_off : tab_off + 16 * max_tiles].view(np.int32).reshape(max_tiles, 4)
    ends = np.cumsum(counts)
    starts = ends - counts
    height = np.zeros(E, np.int64)
    ntiles = np.zeros(E, np.int64)
    for e in range(E):
        c = int(counts[e])
        if c:
            n0 = -(-c // 320)
            height[e] = (-(-c // n0) + 31) // 32 * 32
            ntiles[e] = -(-c // height[e])
    assert count == ntiles.sum()
    assert (tab[count:, 0] == -1).all()
    t = tab[:count]
    assert ((t[:, 0] >= 0) & (t[:, 0] < E)).all()
    ex = t[:, 0]
    assert (t[:, 1] >= starts[ex]).all() and (t[:, 2] <= ends[ex]).all() and (t[:, 1] < t[:, 2]).all()
    assert (t[:, 2] - t[:, 1] <= height[ex]).all()
    cover = np.zeros(M, np.int64)
    for r0, r1 in t[:, 1:3]:
        cover[r0:r1] += 1
    assert (cover == 1).all()
    assert (np.diff(t[:, 1]) > 0).all() and (np.diff(ex) >= 0).all(), "tiles out of expert / row order"
    for e in np.unique(ex):
        idx = np.nonzero(ex == e)[0]
        assert (t[idx[:-1], 2] - t[idx[:-1], 1] == height[e]).all()
    ref = _gmm_ref(to_np(x), to_np(w), counts)
    assert_close(to_np(out), ref, TOL, "to_np(out)")


def test_probe_times_one_gemm_kernel(ops):
    """The timing probe brackets exactly the next forward GEMM launch: its
    span lies inside the op's own event span, and the probe disarms after
    one launch (a second op leaves the events untouched)."""
    rng = np.random.default_rng(5)
    M, E, N, K = 4096, 8, 512, 1024
    counts = _counts("random", M, E, rng)
    x, w, offs = bf16_dev(rand_bf16(rng, (M, K))), bf16_dev(rand_bf16(rng, (E, N, K), 0.05)), _offs(counts)
    announce("probe_next_gemm")
    ops.grouped_mm(x, w, offs)  # warm
    p0, p1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    o0, o1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    ops.probe_next_gemm(p0, p1)
    o0.record()
    out = ops.grouped_mm(x, w, offs)
    o1.record()
    torch.cuda.synchronize()
    probe_ms, op_ms = p0.elapsed_time(p1), o0.elapsed_time(o1)
    assert 0.0 < probe_ms <= op_ms
    assert_close(to_np(out), _gmm_ref(to_np(x), to_np(w), counts), TOL, "to_np(out)")
    # disarmed: the next op does not record the probe events again
    marker = torch.cuda.Event(enable_timing=True)
    marker.record()
    ops.grouped_mm(x, w, offs)
    torch.cuda.synchronize()
    assert p1.elapsed_time(marker) > 0.0
    with pytest.raises(ValueError):
        ops.probe_next_gemm(p0, None)



# Output-tile counts that leave a partial last round of the persistent walk
# on 256 CUs, with enough rows for the tail split to cut the leftover tiles
# along the rows: one expert over 2048 rows (300 tiles: 44 left over, 4
# pieces of 8 stages), and three experts whose leftover tiles belong to a
# loaded expert (2 pieces of 11 stages) or to an expert without rows.
WGRAD_SPLIT_CASES = [
    ([2048], 3840, 5120),
    ([1900, 0, 1400], 2560, 2560),
    ([1900, 1400, 0], 2560, 2560),
]


@pytest.mark.parametrize("counts,N,K", WGRAD_SPLIT_CASES)
def test_grouped_mm_wgrad_tail_split(ops, counts, N, K):
    """The leftover output tiles of a walk that ends in a partial round are
    cut along the expert's rows into pieces summed in piece order: against
    the oracle per expert slice, bit-identical on a second call (whichever
    piece arrives last), exact zeros for an expert without rows, and (fp32)
    not bit-identical to the unsplit kernel, so the pieces did run."""
    import ctypes

    from gpu_util import assert_close

    lib = importlib.import_module("torchtitan-ascend_amd._lib")
    counts = np.array(counts)
    M, E = int(counts.sum()), counts.size
    rng = np.random.default_rng(M + N + K)
    dy = rand_bf16(rng, (M, N))
    x = rand_bf16(rng, (M, K))
    ref = O.grouped_wgrad(dy, x, np.cumsum(counts), E)
    dyd, xd, offs = bf16_dev(dy), bf16_dev(x), _offs(counts)
    for out_dtype in (torch.float32, torch.bfloat16):
        announce(f"wgrad tail split counts={counts.tolist()} N={N} K={K} {out_dtype}")
        a = ops.grouped_mm_wgrad(dyd, xd, offs, E, out_dtype)
        b = ops.grouped_mm_wgrad(dyd, xd, offs, E, out_dtype)
        torch.cuda.synchronize()
        assert torch.equal(a, b), "split sums differ between calls"
        got = to_np(a)
        for e in np.where(counts == 0)[0]:
            assert not np.any(got[e]), f"expert {e} has no rows but a nonzero gradient"
        assert_close(got, ref, TOL, f"wgrad split {out_dtype}")
        if out_dtype == torch.float32:
            plain = torch.empty_like(a)
            lib.call("ttamd_grouped_mm_wgrad", ctypes.c_void_p(dyd.data_ptr()), ctypes.c_void_p(xd.data_ptr()),
                     ctypes.c_void_p(offs.data_ptr()), M, E, N, K, ctypes.c_void_p(plain.data_ptr()), 1, None, 0,
                     ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
            torch.cuda.synchronize()
            assert_close(to_np(plain), ref, TOL, "wgrad unsplit")
            if counts[-1] > 0:
                assert not torch.equal(a, plain), "the tail split did not run"
