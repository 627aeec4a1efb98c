"""The GEMV's two shapes (four waves of 16 columns, all of K; eight waves over
16 columns) at the ends of their ranges: fewer columns than a wave, groups left
over after the waves' unrolled walk, rows 1 to 8, a biased dense call."""
import numpy as np
import pytest

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
