"""A block's q, k and v as one launch (by the rounds of the chip): each with the
bits of its own launch, so the block equals its public calls one by one, over
the tile heights (64 to 256 rows, 256-row rounds followed by a lower height) and
the K split. The launch counts show that the merged route ran."""
import numpy as np
import pytest

import test_block_gpu as tb
from helpers import (bf16, build_block, from_dev, make_lora, merged_split_rows, randn,
                     split_plan)

pytestmark = pytest.mark.gpu
BUCKET = {4: "qproj_fast.w4", 8: "qproj_fast.w8", 16: "qproj.dense"}


# H = 512 (no K split): six column tiles in the merged launch, the heights of 1000
# to 11000 rows. H = 1024 splits K in two, in 64- and 128-row tiles.
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
    _equals_its_calls(ctx, gp, desc, bits, Hd, rows)


def _equals_its_calls(ctx, gp, desc, bits, Hd, rows):
    """The block with its q, k and v merged against its public calls."""
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


# The merged split in 256-row tiles, as the caption block's 203 rows take it.
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("Hd,rows", [(1024, 1360), (3840, 203)])
def test_merged_split_high_tiles(ctx, monkeypatch, bits, Hd, rows):
    slices = split_plan(rows, Hd, Hd)[0]
    assert slices >= 2 and merged_split_rows(rows, Hd, Hd, slices) == 256
    test_merged_qkv_bits(ctx, monkeypatch, bits, Hd, rows)


# q, k and v with different adapters: a tail of its own each (k a longer one, v
# none, dense one of 32 ranks), which also moves each one's K slices.
@pytest.mark.parametrize("bits,Hd,rows", [(4, 512, 1000), (8, 512, 3000), (16, 512, 1000),
                                          (4, 1024, 203), (8, 1024, 700)])
def test_merged_different_adapters(ctx, monkeypatch, bits, Hd, rows):
    print(f"case merged adapters bits={bits} H={Hd} rows={rows}", flush=True)
    monkeypatch.setattr(tb, "H", Hd)
    monkeypatch.setattr(tb, "NH", Hd // 128)
    _, gp, desc = build_block(ctx, 975, Hd, tb.F, tb.ADA, bits, False)
    assert tb.SCALES[0] and tb.SCALES[3]
    gp["k"].bind_lora(0, *make_lora(976, Hd, Hd, 100))
    # a dense v without any might split K by itself, apart from the others
    for slot in (0, 3) if bits != 16 else (3,):
        gp["v"].unbind_lora(slot)
    _equals_its_calls(ctx, gp, desc, bits, Hd, rows)
