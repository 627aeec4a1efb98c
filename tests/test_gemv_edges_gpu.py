"""The GEMV's shapes (four or eight waves over 16 or 32 columns, K split over
them) at the ends of their ranges: fewer columns than a wave, groups left
over after the waves' unrolled walk, rows 1 to 8, a biased dense call."""
import ctypes as C

import numpy as np
import pytest
import torch

import ming_dit_amd as m
from helpers import bf16, empty_bf16, from_dev, make_weight, randn, sync, to_dev

pytestmark = pytest.mark.gpu


def _close(orc, got, ref):
    """Every element within its one bf16 rounding (half an ulp: at most 2^-8 of
    it) and the f32 sums' error (K <= 4160 terms of one sign pattern: below 1e-4
    of the largest result). The mean bar of the other tests needs more elements
    than eight."""
    got = orc.bf16_to_f32(from_dev(got)).astype(np.float64)
    assert (np.abs(got - ref) <= 2.0 ** -8 * np.abs(ref) + 1e-4 * np.abs(ref).max()).all()


@pytest.mark.parametrize("bits", [4, 8, 16])
@pytest.mark.parametrize("M,N,K", [(1, 8, 64), (8, 24, 256), (3, 72, 128), (5, 40, 320),
                                   (7, 136, 2112), (2, 72, 4160), (8, 1000, 512)])
def test_gemv_edges(ctx, orc, bits, M, N, K):
    print(f"case gemv bits={bits} M={M} N={N} K={K}", flush=True)
    x = bf16(randn(9950 + M, (M, K)))
    pack, w = make_weight(9960 + N, N, K, bits)
    qw = (m.QWeight.dense(ctx, pack["w"]) if bits == 16 else
          m.QWeight.quantized(ctx, pack["codes"], pack["scales"], pack["biases"], bits))
    xd, y = to_dev(x), empty_bf16(M, N)
    ref = orc.proj(x, w)
    sync()
    e0 = ctx.engagement()["gemv"]
    ctx.lin(qw, xd, y, M)
    sync()
    assert ctx.engagement()["gemv"] == e0 + 1
    _close(orc, y, ref)
    if bits == 16:
        b = bf16(randn(9970, (N,)))
        ctx.lin_bias(qw, xd, y, M, to_dev(b))
        sync()
        _close(orc, y, ref + orc.bf16_to_f32(b)[None])
    # a row's bits do not depend on the rows beside it
    z = empty_bf16(1, N)
    ctx.lin(qw, xd[M - 1:], z, 1)
    ctx.lin(qw, xd, y, M)
    sync()
    assert np.array_equal(from_dev(y)[M - 1], from_dev(z)[0])
    qw.close()


# Four or eight classes of groups (K to 512 and past it), 16 columns a block or
# 32 (more than 12288 of them), and the last block's second half past N.
@pytest.mark.parametrize("bits", [4, 8, 16])
@pytest.mark.parametrize("M,N,K", [(1, 24, 512), (4, 40, 576), (1, 12296, 192), (8, 12328, 448),
                                   (2, 12296, 576), (1, 12312, 1152)])
def test_gemv_shapes(ctx, orc, bits, M, N, K):
    test_gemv_edges(ctx, orc, bits, M, N, K)


class _Args(C.Structure):
    _fields_ = [("x", C.c_void_p), ("ldx", C.c_longlong), ("codes", C.c_void_p),
                ("sb", C.c_void_p), ("w16", C.c_void_p), ("y", C.c_void_p),
                ("ldy", C.c_longlong), ("M", C.c_int), ("N", C.c_int), ("K", C.c_int),
                ("bias", C.c_void_p)]


class _Batch(C.Structure):
    _fields_ = [("base", _Args), ("count", C.c_int), ("e", (C.c_void_p * 4) * 32)]


@pytest.mark.parametrize("bits", [4, 8, 16])
@pytest.mark.parametrize("N,K,count", [(8, 64, 1), (40, 256, 3), (1032, 512, 2), (72, 576, 3),
                                       (12296, 320, 2), (264, 2112, 32)])
def test_gemv_batch_bits(ctx, bits, N, K, count):
    """An entry of a batched launch (a forward's adaLN projections) has the bits
    of the single launch: mirrors GemvArgs and GemvBatch (kernels.h), weights in
    the resident layout."""
    print(f"case gemv batch bits={bits} N={N} K={K} count={count}", flush=True)
    single, batch = (getattr(m.lib(), s) for s in (
        "_ZN4ming11launch_gemvEiRKNS_8GemvArgsEP12ihipStream_t",
        "_ZN4ming17launch_gemv_batchEiRKNS_9GemvBatchEP12ihipStream_t"))
    single.argtypes = batch.argtypes = [C.c_int, C.c_void_p, C.c_void_p]
    rng = np.random.default_rng(9980 + N)
    x = to_dev(bf16(randn(9981, (1, K))))
    sb, w16, codes, y, z = [], [], [], empty_bf16(count, N), empty_bf16(count, N)
    for i in range(count):
        s, b = bf16(np.abs(randn(9982 + i, (K // 64, N), 0.01))), bf16(randn(9990 + i, (K // 64, N)))
        sb.append(to_dev(np.stack([s, b], -1)))
        w16.append(to_dev(bf16(randn(10000 + i, (N, K)))))
        codes.append(to_dev(rng.integers(0, 1 << 16, (N, K * bits // 16)).astype(np.uint16)))
    st = torch.cuda.current_stream().cuda_stream
    b = _Batch()
    b.base = _Args(x.data_ptr(), K, None, None, None, None, N, 1, N, K, None)
    b.count = count
    sync()
    for i in range(count):
        p = (codes[i].data_ptr(), sb[i].data_ptr(), w16[i].data_ptr())
        a = _Args(x.data_ptr(), K, *p, y[i].data_ptr(), N, 1, N, K, None)
        assert single(bits, C.byref(a), st) == 0
        b.e[i] = (C.c_void_p * 4)(*p, z[i].data_ptr())
    assert batch(bits, C.byref(b), st) == 0
    sync()
    assert np.array_equal(from_dev(y), from_dev(z))
