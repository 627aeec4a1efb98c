"""The pack quantizer at group counts off its 64-group blocks, a source that is
not 16-byte aligned, and groups of zeros, signed zeros and one constant: codes,
scales and biases bit for bit the oracle's recipe."""
import numpy as np
import pytest
import torch

import ming_dit_amd as m  # noqa: F401
from helpers import randn, sync

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offset", [0, 1, 2])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("N,K", [(1, 64), (3, 192), (7, 640), (64, 64), (65, 1088)])
def test_quantize_groups(ctx, orc, bits, N, K, offset):
    w = randn(9900 + N + K, (N, K), 0.02)
    w[0, :64] = 0.0
    if N > 2:
        w[1, :64] = 0.25
        w[2, :64:2], w[2, 1:64:2] = 0.0, -0.0
    buf = torch.empty(N * K + 4, dtype=torch.float32, device="cuda")
    wd = buf[offset:offset + N * K]
    wd.copy_(torch.from_numpy(w.reshape(-1)))
    codes = torch.empty((N, K * bits // 32), dtype=torch.int32, device="cuda")
    sc, bi = (torch.empty((N, K // 64), dtype=torch.int16, device="cuda") for _ in range(2))
    sync()
    ctx.quantize_pack(wd, N, K, bits, codes, sc, bi)
    sync()
    c, s, b = orc.quantize(w, bits)
    assert np.array_equal(codes.cpu().numpy().view(np.uint32), c)
    assert np.array_equal(sc.cpu().numpy().view(np.uint16), s)
    got, want = bi.cpu().numpy().view(np.uint16), b
    # the least of a group of +0 and -0 may carry either sign
    assert np.array_equal(np.where(got == 0x8000, 0, got), np.where(want == 0x8000, 0, want))
