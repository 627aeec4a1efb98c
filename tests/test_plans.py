"""The launch plans, which choose tile heights and K slices by size alone: on the
CPU (without a device they count the MI355X's 256 CUs), through the library's
own symbols."""
import pytest

from helpers import dense_plan, plan_rows, xa_tile

SHAPES = [(M, tn, st) for M in (1, 63, 300, 700, 1280, 2085, 4352, 8320, 16640)
          for tn in (1, 8, 15, 40, 60, 80, 129) for st in (1, 4, 16, 60, 165)]


@pytest.mark.parametrize("pair", [False, True])
def test_row_plans_cover_the_rows(pair):
    for M, tn, st in SHAPES:
        p = plan_rows(M, tn, st, pair)
        assert p.rows_main == M or (p.rows_main % 256 == 0 and 0 <= p.rows_main < M), (M, tn, st)
        assert p.rf_rest in ((8, 6, 4) if pair else (8, 6, 4, 2)), (M, tn, st)


def test_row_plans_count_k():
    """A short K leaves a second launch little to gain for its start: plans that
    are two launches at K = 3840 are one at K = 64."""
    two = [s for s in ((5600, 40), (8320, 40), (16640, 40)) if 0 < plan_rows(*s, 60, False).rows_main < s[0]]
    assert two
    for M, tn in two:
        assert plan_rows(M, tn, 1, False).rows_main in (0, M)
    # 4096 rows of [10240, 64]: one launch of a lower height (28.5 us, 36.2 as
    # 256-row tiles and then 192)
    assert plan_rows(4096, 40, 1, False).rows_main == 0
    # 2560 rows of [10240, 3840]: one launch of 256-row tiles (171.8 us, 178.2)
    assert plan_rows(2560, 40, 60, False).rows_main == 2560
    # a paired launch's 4352 rows: five whole rounds, then 128-row tiles
    p = plan_rows(4352, 80, 60, True)
    assert (p.rows_main, p.rf_rest) == (4096, 4)


@pytest.mark.parametrize("M,N,K", [(203, 10240, 256), (1024, 3840, 64), (130, 15360, 128),
                                   (1024, 2560, 256), (40, 10240, 64), (16, 64, 64)])
def test_dense_plans_of_a_short_k(M, N, K):
    """A tall tile's scattered stores are most of an unsplit launch of a few K
    stages: 203 rows of [10240, 256] take 13.2 us on 256 x 128, 7.4 on the dense
    route."""
    rows, cols, slices = dense_plan(M, N, K)
    assert slices == 0 or rows * cols <= 128 * 64


def test_xa_tiles_at_half_a_chip():
    """The adapters' x.A: 256 x 128 tiles from half a chip of them on (512 ranks at
    8320 rows: 65 us, 64-row tiles 74), a block more where K is short."""
    assert xa_tile(8320, 512, 3840, 1) == (256, 128)
    assert xa_tile(16640, 256, 10240, 1) == (256, 128)
    assert xa_tile(16640, 256, 3840, 1) == (64, 128)
    assert xa_tile(16384, 256, 10240, 1) == (64, 128)
    assert xa_tile(4352, 64, 3840, 3) == (64, 64)
