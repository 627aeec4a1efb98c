"""The residual norms of a block at few rows (a row a block, up to 2048 rows of
520 to 4096 columns) give the bits of the public rmsnorm, residual and gated
residual one by one, as the many-row form does: widths of both register counts,
rows around a wave, a block and the limit."""
import numpy as np
import pytest

import test_block_gpu as tb
from helpers import bf16, build_block, from_dev, randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("modulated", [True, False])
@pytest.mark.parametrize("Hd,rows", [(640, 1), (640, 133), (640, 2048), (640, 2049), (2176, 3),
                                     (2176, 130)])
def test_residual_norm_rows(ctx, monkeypatch, modulated, Hd, rows):
    print(f"case residual norms H={Hd} rows={rows} modulated={modulated}", flush=True)
    monkeypatch.setattr(tb, "H", Hd)
    monkeypatch.setattr(tb, "NH", Hd // 128)
    _, gp, desc = build_block(ctx, 980, Hd, tb.F, tb.ADA, 4, modulated)
    x = bf16(randn(981, (rows, Hd)))
    temb = bf16(randn(982, (tb.ADA,))) if modulated else None
    c, s = tb.tables(rows)
    got = tb.run_gpu(ctx, desc, tb.dims(), x, rows, c, s, temb, tb.SCALES)
    xd, nrm, qkv, ob, ffg, _, mods = tb.public_block(ctx, gp, x, rows, c, s, temb, tb.SCALES,
                                                     modulated)
    ctx.ffn(gp["w1"], gp["w3"], gp["w2"], nrm, ob, rows, tb.SCALES, h=ffg)
    ctx.rmsnorm(ob, gp["fn2"], ob, rows, Hd)
    if modulated:
        ctx.gated_residual(xd, mods[:, 3 * Hd:], ob, rows, Hd)
    else:
        ctx.residual_add(xd, ob, rows, Hd)
    ctx.synchronize()
    assert np.array_equal(got, from_dev(xd))
    for q in gp.values():
        if hasattr(q, "close"):
            q.close()
