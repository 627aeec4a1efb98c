"""The dense bf16 route (dense_fast.hip) over its tile heights, ring
remainders and tails: against the oracle at the projection bar (2e-3, the
output's one bf16 rounding being 1.66e-3), and bit for bit against the general
kernel, which multiplies in the same k16 order and rounds once too."""
import numpy as np
import pytest

import ming_dit_amd as m
from helpers import bf16, dense_plan, empty_bf16, from_dev, make_lora, make_weight, randn, sync, to_dev

pytestmark = pytest.mark.gpu
TOL = 2e-3


def _run(ctx, route, fn, M, N, ldy=None):
    ctx.set_route(route)
    y = empty_bf16(M, ldy or N)
    y.zero_()
    sync()
    fn(y)
    sync()
    ctx.set_route("auto")
    return from_dev(y)


# N % 64 != 0 (or a live adapter) keeps a small grid off the split-K GEMM.
# 64-row tiles while they fit one round of 256 blocks, taller ones past it.
@pytest.mark.parametrize("M,N,K,ranks", [
    (9, 264, 64, ()),                  # one stage, one ragged row tile
    (65, 264, 128, (8,)),              # two stages; an odd tail of one chunk
    (200, 1000, 192, (32, 32)),        # a tail of two chunks, ragged columns
    (130, 520, 320, (4, 40, 64)),      # five stages; four chunks
    (2085, 2056, 384, (16, 64)),       # 128-row tiles; three chunks
    (4300, 2048, 448, (64, 64, 48)),   # 192-row tiles; six chunks, seven stages
    (6210, 2048, 256, (33,)),          # 256-row tiles; two chunks
])
def test_dense_route(ctx, orc, M, N, K, ranks):
    print(f"case dense M={M} N={N} K={K} ranks={ranks}", flush=True)
    x = bf16(randn(9000 + M, (M, K)))
    pack, w = make_weight(9100 + N, N, K, 16, std=1.0 / np.sqrt(K))
    qw = m.QWeight.dense(ctx, pack["w"])
    scales, loras = [0.0] * 8, []
    for i, r in enumerate(ranks):
        A, B = make_lora(9200 + 2 * i, N, K, r)
        qw.bind_lora(i, A, B)
        scales[i] = 0.7 - 0.4 * i
        loras.append((A, B, scales[i]))
    xd = to_dev(x)
    got, want = (_run(ctx, r, lambda y: ctx.lin(qw, xd, y, M, scales), M, N)
                 for r in ("auto", "general"))
    ref = orc.proj(x, w, loras)
    assert orc.rel_l2(orc.bf16_to_f32(got), ref) <= TOL
    if ranks:
        # the two routes slice the x.A differently: T may differ by a bf16 ulp
        assert orc.rel_l2(orc.bf16_to_f32(got), orc.bf16_to_f32(want)) <= 1e-3
        got, want = (_run(ctx, r, lambda y: ctx.lin(qw, xd, y, M), M, N)
                     for r in ("auto", "general"))
    assert np.array_equal(got, want)
    # the fused bias and SwiGLU, and an output stride that leaves 8-byte rows
    bias, gate = to_dev(bf16(randn(9300, (N,)))), to_dev(bf16(randn(9301, (M, N))))
    for ldy, fn in ((N, lambda y: ctx.lin_bias(qw, xd, y, M, bias)),
                    (N, lambda y: ctx.lin_swiglu(qw, xd, gate, y, M)),
                    (N + 4, lambda y: ctx.lin(qw, xd, y, M, ldy=N + 4))):
        a, b = (_run(ctx, r, fn, M, N, ldy) for r in ("auto", "general"))
        assert np.array_equal(a, b)
    qw.close()


@pytest.mark.parametrize("M", [40, 300])
def test_dense_gated_few_tiles(ctx, M):
    """A gated dense projection of few tiles gives ming_lin's bits, then
    ming_swiglu's, whichever kernel ming_lin takes."""
    N, K = 512, 2048
    pack, _ = make_weight(9400, N, K, 16, std=1.0 / np.sqrt(K))
    qw = m.QWeight.dense(ctx, pack["w"])
    xd, g = to_dev(bf16(randn(9401, (M, K)))), to_dev(bf16(randn(9402, (M, N))))
    u, want, got = empty_bf16(M, N), empty_bf16(M, N), empty_bf16(M, N)
    sync()
    ctx.lin(qw, xd, u, M)
    ctx.swiglu(g, u, want, M, N)
    ctx.lin_swiglu(qw, xd, g, got, M)
    sync()
    assert np.array_equal(from_dev(got), from_dev(want))
    qw.close()


# The output in x's own memory: no wider than x, and wider at a stride past both.
@pytest.mark.parametrize("M,N,K,ld", [(600, 1032, 1088, 1088), (2100, 2056, 2112, 2112),
                                      (300, 1032, 576, 1664)])
def test_dense_gated_over_x(ctx, M, N, K, ld):
    pack, _ = make_weight(9410, N, K, 16, std=1.0 / np.sqrt(K))
    qw = m.QWeight.dense(ctx, pack["w"])
    xd, g = to_dev(bf16(randn(9411, (M, ld)))), to_dev(bf16(randn(9412, (M, N))))
    want = empty_bf16(M, N)
    sync()
    ctx.lin_swiglu(qw, xd, g, want, M, ldx=ld)
    ctx.lin_swiglu(qw, xd, g, xd, M, ldx=ld, ldo=ld)
    sync()
    assert np.array_equal(from_dev(xd)[:, :N], from_dev(want))
    qw.close()


# Tiles of 128 x 64 and 128 x 128, one slice and several, more columns than the
# adapters' group table holds.
@pytest.mark.parametrize("M,N,K", [(9, 4160, 1024), (17, 256, 4096), (130, 1984, 640),
                                   (231, 1024, 2560), (300, 3840, 1024), (500, 704, 6400)])
def test_dense_few_tiles(ctx, orc, M, N, K):
    print(f"case dense split M={M} N={N} K={K}", flush=True)
    x = bf16(randn(9800 + M, (M, K)))
    pack, w = make_weight(9801 + N, N, K, 16, std=1.0 / np.sqrt(K))
    b = bf16(randn(9802, (N,)))
    qw = m.QWeight.dense(ctx, pack["w"])
    xd, bd = to_dev(x), to_dev(b)
    ref = orc.proj(x, w)
    plain = _run(ctx, "auto", lambda y: ctx.lin(qw, xd, y, M), M, N)
    biased = _run(ctx, "auto", lambda y: ctx.lin_bias(qw, xd, y, M, bd), M, N)
    assert orc.rel_l2(orc.bf16_to_f32(plain), ref) <= TOL
    assert orc.rel_l2(orc.bf16_to_f32(biased), ref + orc.bf16_to_f32(b)[None]) <= TOL
    # slices are summed in order: the same bits again
    assert np.array_equal(plain, _run(ctx, "auto", lambda y: ctx.lin(qw, xd, y, M), M, N))
    qw.close()


# Every tile of the plan, split and not (64 x 128 and 256 x 128 only split: unsplit
# the plan finds others faster).
@pytest.mark.parametrize("M,N,K,tile,split", [
    (700, 1536, 192, (64, 64), False), (9, 4160, 10240, (64, 128), True),
    (17, 1216, 640, (128, 64), False), (231, 832, 3840, (128, 64), True),
    (1500, 2240, 1024, (128, 128), False), (9, 2112, 2560, (128, 128), True),
    (130, 832, 10240, (256, 128), True), (4096, 256, 3840, (256, 128), True)])
def test_dense_plan_tiles(ctx, orc, M, N, K, tile, split):
    rows, cols, slices = dense_plan(M, N, K)
    assert (rows, cols) == tile and (slices > 1 if split else slices == 1)
    test_dense_few_tiles(ctx, orc, M, N, K)


@pytest.mark.parametrize("M,K", [(70, 256), (2100, 640)])
def test_dense_segments(ctx, M, K):
    """A concatenated dense weight, its segments with adapters of their own and
    none, gives each part's own bits (64- and 192-row tiles)."""
    print(f"case dense segments M={M} K={K}", flush=True)
    parts, Ns, ranks = [], (256, 512, 1032), ((16, 64), (), (40,))
    for i, N in enumerate(Ns):
        q = m.QWeight.dense(ctx, make_weight(10400 + i, N, K, 16, std=1.0 / np.sqrt(K))[0]["w"])
        for s, r in enumerate(ranks[i]):
            q.bind_lora(s, *make_lora(10410 + 2 * (4 * i + s), N, K, r))
        parts.append(q)
    fused = m.QWeight.concat(ctx, parts)
    assert fused.n_segments == 3
    xd, sc = to_dev(bf16(randn(10450, (M, K)))), [0.7, -0.4] + [0.0] * 6
    got = _run(ctx, "auto", lambda y: ctx.lin(fused, xd, y, M, sc), M, sum(Ns))
    general = _run(ctx, "general", lambda y: ctx.lin(fused, xd, y, M, sc), M, sum(Ns))
    n0 = 0
    for i, N in enumerate(Ns):
        want = _run(ctx, "auto", lambda y: ctx.lin(parts[i], xd, y, M, sc), M, N)
        mine = got[:, n0:n0 + N]
        if ranks[i]:
            assert np.array_equal(mine, want)
        else:
            # alone, with no adapter, the part may split K
            assert np.array_equal(mine, general[:, n0:n0 + N])
        n0 += N
    for q in parts + [fused]:
        q.close()
