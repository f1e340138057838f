"""How many splits of the key range a decode step's chain takes (a rule on the host)."""
import pytest

from rocml_amd import ops


@pytest.mark.parametrize("pages,pairs,splits", [
    (1, 8, 1), (4, 32, 1), (8, 8, 4), (8, 32, 4), (64, 8, 32), (32, 16, 16), (16, 32, 8), (16, 24, 8),      # two pages a split, at most 256 items
    (128, 8, 20), (64, 16, 10), (32, 32, 5), (32, 24, 6), (1024, 8, 20), (1024, 1, 64), (64, 512, 1)])      # beyond: some 160 items
def test_splits(pages, pairs, splits):
    assert ops.decode_chain_splits(pages, pairs) == splits
