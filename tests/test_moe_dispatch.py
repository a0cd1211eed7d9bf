"""From how many rows an expert the grouped products run on the 256-row tile."""
import pytest

from omnia_amd import ops


@pytest.mark.parametrize("rows", [0, 64, 128, 512])
def test_the_flag_sets_the_tiles_first_rows(rows, monkeypatch):
    """OMNIA_MOE_TILE256_ROWS is the line for every size, below the measured ones too."""
    monkeypatch.setattr(ops, "MOE_TILE256_ROWS", rows)
    assert {ops.moe_tile_rows(e, d) for e in (1, 8, 64) for d in (256, 2048, 4096)} == {rows}


def test_unset_it_lies_by_the_down_products_tiles(monkeypatch):
    monkeypatch.setattr(ops, "MOE_TILE256_ROWS", None)
    assert [ops.moe_tile_rows(8, d) for d in (2048, 4064, 4096)] == [224, 224, 128]
