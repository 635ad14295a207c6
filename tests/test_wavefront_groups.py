"""Blocks of two and four groups of wavefronts that share a tile's slabs (launch plans 16-18, statistics tiles 8-10): what the other
plans' tests ask of them, at the same shapes (partial tiles, fewer slabs than groups, remainders, infinities, lost bits)."""
import pytest

from tests import test_parity_conv as conv
from tests import test_split_products as split

pytestmark = pytest.mark.gpu
PLANS = pytest.mark.parametrize("plan", [16, 17, 18])


@PLANS
@pytest.mark.parametrize("dims", split.REDO_SHAPES + [(1, 80, 9, 9, 70, 1, 1, 1, 1, 0, 0), (2, 272, 7, 7, 68, 1, 1, 1, 1, 0, 0)], ids=lambda d: "x".join(map(str, d)))
def test_what_the_terms_cannot_hold(on_hip, dims, plan, monkeypatch):
    if dims[0] == 1:
        dims = (2,) + dims[1:]          # (the values are planted in the second sample)
    split.test_what_the_terms_cannot_hold_under_every_launch_plan(on_hip, dims, plan, monkeypatch)


@PLANS
@pytest.mark.parametrize("dims", conv.SHARED_TAIL_SHAPES, ids=lambda d: "x".join(map(str, d)))
def test_against_whole_tiles_and_twice(on_hip, dims, plan, monkeypatch):
    conv.test_whole_tiles_and_slices_of_the_last_ones(on_hip, dims, plan, monkeypatch)


@pytest.mark.parametrize("tile", [8, 9, 10])
def test_statistics_of_small_rows(on_hip, tile, monkeypatch):
    split.test_small_filter_rows_with_the_statistics_of_their_outputs(on_hip, tile, monkeypatch)
