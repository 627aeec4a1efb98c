"""Projections under stream capture: what a captured call needs of the context's
scratch, and what stays of it for the graph's replays when a later call grows
it. Every replay is checked against the eager call, with eager work between."""
import ctypes as C

import numpy as np
import pytest
import torch

import ming_dit_amd as m
import test_block_gpu as tb
from helpers import (bf16, build_block, empty_bf16, from_dev, make_weight, randn, split_plan, sync,
                     to_dev)

pytestmark = pytest.mark.gpu


@pytest.fixture()
def cap():
    """A context of its own (cold scratch) on a stream that can be captured."""
    s = torch.cuda.Stream()
    c = m.Ctx(0, s.cuda_stream)
    c.stream = s
    yield c
    c.close()


def _weight(ctx, seed, N, K, bits):
    pack, _ = make_weight(seed, N, K, bits, std=1.0 / np.sqrt(K))
    if bits == 16:
        return m.QWeight.dense(ctx, pack["w"])
    return m.QWeight.quantized(ctx, pack["codes"], pack["scales"], pack["biases"], bits)


def _capture(ctx, fn):
    sync()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=ctx.stream, capture_error_mode="thread_local"):
        fn()
    return g


def test_growth_after_a_capture_keeps_the_graphs_scratch(cap):
    """A split projection captured with a small partials' buffer still replays
    to its own bits, into memory of its own, after a larger call grew it."""
    M, N, K = 40, 512, 2048
    q, big = _weight(cap, 4000, N, K, 4), _weight(cap, 4001, 3840, 3840, 4)
    x = [to_dev(bf16(randn(4002 + i, (M, K)))) for i in range(3)]
    xb, yb = to_dev(bf16(randn(4005, (256, 3840)))), empty_bf16(256, 3840)
    xi, y = empty_bf16(M, K), empty_bf16(M, N)
    sync()
    want = []
    for v in x:
        cap.lin(q, v, y, M)
        cap.synchronize()
        want.append(from_dev(y))
    cap.reset_engagement()
    g = _capture(cap, lambda: cap.lin(q, xi, y, M))
    assert cap.engagement()["gemm_split"] == 1
    cap.lin(big, xb, yb, 256)                     # about 16 MB of partials
    cap.synchronize()
    first = from_dev(yb)
    other = [torch.full((1 << 18,), 7, dtype=torch.int32, device="cuda") for _ in range(8)]
    for v, w in zip(x, want):
        xi.copy_(v)
        y.zero_()
        sync()
        g.replay()
        sync()
        assert np.array_equal(from_dev(y), w)
        cap.lin(big, xb, yb, 256)
        cap.synchronize()
        assert np.array_equal(from_dev(yb), first)
    assert all(bool((o == 7).all()) for o in other)
    del g
    q.close()
    big.close()


def _cap_partials(ctx, nbytes):
    f = m.lib()._ZN4ming15rt_set_part_capEP8ming_ctxm
    f.argtypes, f.restype = [C.c_void_p, C.c_size_t], None
    f(ctx.h, nbytes)


@pytest.mark.parametrize("M,N,K,gated", [(203, 10240, 3840, False), (17, 4160, 1024, False),
                                         (40, 1024, 2560, False), (130, 4160, 2048, True)])
def test_dense_split_gives_way(orc, cap, M, N, K, gated):
    """A dense projection of few rows that splits K runs unsplit, on the dense
    route, where its partials have no room: under capture in a cold context,
    and without memory for them."""
    x, g = bf16(randn(4100 + M, (M, K))), bf16(randn(4101, (M, N)))
    pack, w = make_weight(4102 + N, N, K, 16, std=1.0 / np.sqrt(K))
    q = m.QWeight.dense(cap, pack["w"])
    xd, gd, y = to_dev(x), to_dev(g), empty_bf16(M, N)
    call = (lambda: cap.lin_swiglu(q, xd, gd, y, M)) if gated else (lambda: cap.lin(q, xd, y, M))
    graph = _capture(cap, call)
    seen = []
    for _ in range(3):
        y.zero_()
        sync()
        graph.replay()
        sync()
        seen.append(from_dev(y))
    assert np.array_equal(seen[0], seen[1]) and np.array_equal(seen[0], seen[2])
    _cap_partials(cap, 0)
    call()
    cap.synchronize()
    assert np.array_equal(from_dev(y), seen[0])
    _cap_partials(cap, 1 << 40)
    call()
    cap.synchronize()
    ref = orc.proj(x, w)
    if gated:
        ref = orc.bf16_to_f32(orc.swiglu(g, orc.f32_to_bf16(ref)))
    for got in (seen[0], from_dev(y)):
        assert orc.rel_l2(orc.bf16_to_f32(got), ref) <= 2e-3
    graph.replay()
    sync()
    assert np.array_equal(from_dev(y), seen[0])
    del graph
    q.close()


@pytest.mark.parametrize("bits", [4, 8])
def test_merged_split_gives_way(cap, monkeypatch, bits):
    """A block's split q, k and v run as one launch where their partials fit
    together, else (no memory, or captured before they did) as one each with the
    same bits."""
    rows, Hd = 700, 1024
    monkeypatch.setattr(tb, "H", Hd)
    monkeypatch.setattr(tb, "NH", Hd // 128)
    _, gp, desc = build_block(cap, 4200, Hd, tb.F, tb.ADA, bits, False)
    x = bf16(randn(4201, (rows, Hd)))
    c, s = (to_dev(np.ascontiguousarray(t)) for t in tb.tables(rows))
    src, xd = to_dev(x), to_dev(x)
    ws = torch.empty(cap.block_workspace_bytes(tb.dims(), rows), dtype=torch.uint8, device="cuda")
    call = lambda: cap.block_forward(desc, tb.dims(), xd, rows, c, s, None, tb.SCALES, ws)

    def run(go):
        xd.copy_(src)
        sync()
        go()
        cap.synchronize()
        sync()
        return from_dev(xd)

    def launches():
        cap.set_profiling(True)
        got = run(call)
        n = cap.profile_collect()[f"qproj_fast.w{bits}"]["launches"]
        cap.set_profiling(False)
        return got, n

    ks = split_plan(rows, Hd, Hd)[0]
    assert ks >= 2
    _cap_partials(cap, 2 * ks * rows * Hd * 4)      # two projections' partials
    apart, n_apart = launches()
    _cap_partials(cap, 1 << 40)
    graph = _capture(cap, call)                     # the buffer still holds two
    captured = [run(graph.replay) for _ in range(3)]
    merged, n_merged = launches()
    assert n_apart == n_merged + 2
    for got in [merged, run(graph.replay)] + captured:
        assert np.array_equal(got, apart)
    del graph
    for q in gp.values():
        if hasattr(q, "close"):
            q.close()
