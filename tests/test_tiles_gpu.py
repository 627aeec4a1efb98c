"""The quantized route's tile heights (64, 128, 192 and 256 rows, alone and as
256-row rounds followed by a lower height): every output element runs the same
MFMA sequence in each, so a projection over all rows gives the bits of the same
projection over row ranges that take other heights. The all-rows result is held
to the oracle at the projection bar. K < 768 keeps the calls unsplit, K < 1024
the x.A in one slice."""
import numpy as np
import pytest

import ming_dit_amd as m
from helpers import (bf16, empty_bf16, from_dev, make_lora, make_weight, plan_rows, randn,
                     split_plan, sync, to_dev)

pytestmark = pytest.mark.gpu
TOL = 2e-3


def _weight(ctx, seed, N, K, bits, ranks):
    pack, w = make_weight(seed, N, K, bits)
    q = m.QWeight.quantized(ctx, pack["codes"], pack["scales"], pack["biases"], bits)
    loras = []
    for i, r in enumerate(ranks):
        A, B = make_lora(seed + 1 + 2 * i, N, K, r)
        q.bind_lora(i, A, B)
        loras.append((A, B, 0.6 - 0.5 * i))
    return q, w, loras


def _scales(ranks):
    return [0.6 - 0.5 * i for i in range(len(ranks))] + [0.0] * (8 - len(ranks))


# N = 2040: eight column tiles, the last ragged. Rows 1000 take 64-row tiles,
# 2085 128, 4300 and 8250 192, 6210 256.
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,K,ranks", [(1000, 64, ()), (1000, 192, (8, 40)), (2085, 128, (33,)),
                                       (4300, 320, (16, 64)), (6210, 64, (8,)),
                                       (8250, 128, (40,))])
def test_lin_tile_heights(ctx, orc, bits, M, K, ranks):
    N = 2040
    print(f"case tiles bits={bits} M={M} K={K} ranks={ranks}", flush=True)
    q, w, loras = _weight(ctx, 9500 + M, N, K, bits, ranks)
    x = bf16(randn(9501, (M, K)))
    xd, y, z = to_dev(x), empty_bf16(M, N), empty_bf16(M, N)
    sync()
    ctx.lin(q, xd, y, M, _scales(ranks))
    for r in range(0, M, 700):
        ctx.lin(q, xd[r:], z[r:], min(700, M - r), _scales(ranks))
    sync()
    got = from_dev(y)
    assert np.array_equal(got, from_dev(z))
    rows = np.unique(np.r_[0:M:37, M - 1])
    ref = orc.proj(np.ascontiguousarray(x[rows]), w, loras)
    assert orc.rel_l2(orc.bf16_to_f32(np.ascontiguousarray(got[rows])), ref) <= TOL
    q.close()


# F = 1984: sixteen paired column tiles, the last ragged. 300 rows take 128-row
# tiles, 2600 and 4150 192, 4000 256.
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,H,ranks", [(300, 64, (8,)), (2600, 128, (24, 40)), (4000, 128, ()),
                                       (4150, 192, (8,))])
def test_ffn_tile_heights(ctx, bits, M, H, ranks):
    F = 2048 - 64
    print(f"case paired tiles bits={bits} M={M} H={H} ranks={ranks}", flush=True)
    ws = [_weight(ctx, 9600 + i, *s, bits, ranks)[0] for i, s in enumerate(((F, H), (F, H), (H, F)))]
    xd = to_dev(bf16(randn(9601, (M, H))))
    y, h, g, h2 = empty_bf16(M, H), empty_bf16(M, F), empty_bf16(M, F), empty_bf16(M, F)
    sc = _scales(ranks)
    sync()
    e0 = ctx.engagement()["gemm_paired"]
    ctx.ffn(*ws, xd, y, M, sc, h=h)
    assert ctx.engagement()["gemm_paired"] == e0 + 1
    for r in range(0, M, 900):
        n = min(900, M - r)
        ctx.lin(ws[0], xd[r:], g[r:], n, sc)
        ctx.lin_swiglu(ws[1], xd[r:], g[r:], h2[r:], n, sc)
    sync()
    assert np.array_equal(from_dev(h), from_dev(h2))
    for w in ws:
        w.close()


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,N,K,ranks", [(9, 264, 1024, ()), (70, 512, 832, (64, 64, 64, 64)),
                                         (200, 2056, 1600, (32,)), (700, 1032, 4096, (8,)),
                                         (1500, 640, 2048, (128, 128))])
def test_split_tile_heights(ctx, orc, bits, M, N, K, ranks):
    """The split plans of 64-row tiles: two slices and more, the last slice
    shortened by a long tail."""
    print(f"case split bits={bits} M={M} N={N} K={K} ranks={ranks}", flush=True)
    q, w, loras = _weight(ctx, 9700 + M, N, K, bits, ranks)
    x = bf16(randn(9701, (M, K)))
    y = empty_bf16(M, N)
    sync()
    ctx.reset_engagement()
    ctx.lin(q, to_dev(x), y, M, _scales(ranks))
    sync()
    assert ctx.engagement()["gemm_split"] == 1
    assert orc.rel_l2(orc.bf16_to_f32(from_dev(y)), orc.proj(x, w, loras)) <= TOL
    q.close()


def _stages(K, ranks):
    return K // 64 + (sum((r + 7) // 8 * 8 for r in ranks) + 31) // 32 * 5 // 8


# Whole rounds of 256-row tiles, then a lower height at shifted rows: the last
# rows and columns ragged, one adapter and none.
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,N,K,ranks,rf", [(3651, 9976, 320, (), 2), (2584, 14328, 320, (8,), 4),
                                            (2099, 17912, 192, (24,), 6)])
def test_lin_two_heights(ctx, orc, bits, M, N, K, ranks, rf):
    print(f"case two heights bits={bits} M={M} N={N} K={K} ranks={ranks}", flush=True)
    p = plan_rows(M, (N + 255) // 256, _stages(K, ranks), False)
    assert 0 < p.rows_main < M and p.rf_rest == rf
    q, w, loras = _weight(ctx, 10100 + M, N, K, bits, ranks)
    x = bf16(randn(10101, (M, K)))
    xd, y, z = to_dev(x), empty_bf16(M, N), empty_bf16(M, N)
    sync()
    ctx.lin(q, xd, y, M, _scales(ranks))
    for r in range(0, M, 256):
        ctx.lin(q, xd[r:], z[r:], min(256, M - r), _scales(ranks))
    sync()
    got = from_dev(y)
    assert np.array_equal(got, from_dev(z))
    rows = np.unique(np.r_[0:M:113, p.rows_main - 1, p.rows_main, M - 1])
    ref = orc.proj(np.ascontiguousarray(x[rows]), w, loras)
    assert orc.rel_l2(orc.bf16_to_f32(np.ascontiguousarray(got[rows])), ref) <= TOL
    q.close()


# The paired launch the same way.
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,F,H,ranks,rf", [(3651, 9792, 128, (8,), 4), (1323, 9408, 320, (), 6)])
def test_ffn_two_heights(ctx, bits, M, F, H, ranks, rf):
    print(f"case paired two heights bits={bits} M={M} F={F} H={H} ranks={ranks}", flush=True)
    p = plan_rows(M, (F + 127) // 128, _stages(H, ranks), True)
    assert 0 < p.rows_main < M and p.rf_rest == rf
    ws = [_weight(ctx, 10200 + i, *s, bits, ranks)[0]
          for i, s in enumerate(((F, H), (F, H), (H, F)))]
    xd = to_dev(bf16(randn(10201, (M, H))))
    y, h, g, h2 = empty_bf16(M, H), empty_bf16(M, F), empty_bf16(M, F), empty_bf16(M, F)
    sc = _scales(ranks)
    sync()
    e0 = ctx.engagement()["gemm_paired"]
    ctx.ffn(*ws, xd, y, M, sc, h=h)
    assert ctx.engagement()["gemm_paired"] == e0 + 1
    for r in range(0, M, 512):
        n = min(512, M - r)
        ctx.lin(ws[0], xd[r:], g[r:], n, sc)
        ctx.lin_swiglu(ws[1], xd[r:], g[r:], h2[r:], n, sc)
    sync()
    assert np.array_equal(from_dev(h), from_dev(h2))
    for w in ws:
        w.close()


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,N,K,ranks,height", [(700, 3840, 10240, (64,), 256),
                                                (400, 3840, 3840, (64, 64, 64, 64), 128)])
def test_split_high_tiles(ctx, orc, bits, M, N, K, ranks, height):
    """The split plans of 128- and 256-row tiles, with a tail."""
    print(f"case split bits={bits} M={M} N={N} K={K} ranks={ranks}", flush=True)
    slices, rows = split_plan(M, N, K)
    assert slices >= 2 and rows == height
    q, w, loras = _weight(ctx, 10300 + M, N, K, bits, ranks)
    x = bf16(randn(10301, (M, K)))
    y = empty_bf16(M, N)
    sync()
    ctx.reset_engagement()
    ctx.lin(q, to_dev(x), y, M, _scales(ranks))
    sync()
    assert ctx.engagement()["gemm_split"] == 1
    at = np.unique(np.r_[0:M:23, 255, 256, M - 1])
    got = np.ascontiguousarray(from_dev(y)[at])
    ref = orc.proj(np.ascontiguousarray(x[at]), w, loras)
    assert orc.rel_l2(orc.bf16_to_f32(got), ref) <= TOL
    q.close()
