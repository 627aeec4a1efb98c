"""A block's q, k and v as one launch (by the rounds of the chip): each with the
bits of its own launch, so the block equals its public calls one by one, over
the tile heights (64 to 256 rows, 256-row rounds followed by a lower height) and
the K split. The launch counts show that the merged route ran."""
import numpy as np
import pytest

import test_block_gpu as tb
from helpers import bf16, build_block, from_dev, randn

pytestmark = pytest.mark.gpu
BUCKET = {4: "qproj_fast.w4", 8: "qproj_fast.w8", 16: "qproj.dense"}


# H = 512 (no K split): six column tiles in the merged launch. 1000 rows take
# 64-row tiles, 3000 128, 5600 192, 8300 256, 11000 two 256-row rounds and 64
# (dense: 192). H = 1024 splits K in two.
@pytest.mark.parametrize("bits,Hd,rows", [
    (4, 512, 1000), (4, 512, 3000), (4, 512, 5600), (4, 512, 8300), (4, 512, 11000),
    (8, 512, 1000), (8, 512, 8300), (8, 512, 11000),
    (16, 512, 1000), (16, 512, 3000), (16, 512, 5600), (16, 512, 8300),
    (4, 1024, 40), (4, 1024, 700), (4, 1024, 3500), (8, 1024, 40), (8, 1024, 3500)])
def test_merged_qkv_bits(ctx, monkeypatch, bits, Hd, rows):
    print(f"case merged bits={bits} H={Hd} rows={rows}", flush=True)
    monkeypatch.setattr(tb, "H", Hd)
    monkeypatch.setattr(tb, "NH", Hd // 128)
    _, gp, desc = build_block(ctx, 970, Hd, tb.F, tb.ADA, bits, False)
    x = bf16(randn(971, (rows, Hd)))
    c, s = tb.tables(rows)
    ctx.set_profiling(True)
    try:
        got = tb.run_gpu(ctx, desc, tb.dims(), x, rows, c, s, None, tb.SCALES)
        prof = ctx.profile_collect()
    finally:
        ctx.set_profiling(False)
    # q|k|v, o and w2, and w1 and w3 where they are no paired launch
    pairs = prof.get(f"qproj_pair.w{bits}", {}).get("launches", 0)
    assert prof[BUCKET[bits]]["launches"] == 5 - 2 * pairs
    xd, nrm, qkv, ob, ffg, _, _ = tb.public_block(ctx, gp, x, rows, c, s, None, tb.SCALES, False)
    ctx.ffn(gp["w1"], gp["w3"], gp["w2"], nrm, ob, rows, tb.SCALES, h=ffg)
    ctx.rmsnorm(ob, gp["fn2"], ob, rows, Hd)
    ctx.residual_add(xd, ob, rows, Hd)
    ctx.synchronize()
    assert np.array_equal(got, from_dev(xd))
    for q in gp.values():
        if hasattr(q, "close"):
            q.close()
