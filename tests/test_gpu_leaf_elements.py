"""Leaf Grams of the FP64 row trees at the ranks where a lane holds one packed
element (up to 10) and at the first rank of the tiles above: draws with given
uniforms are index-exact against the oracle, as at the tiles' own edges."""
import pytest

import test_gpu_leaf_tiles as leaf_tiles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R", [1, 9, 10, 11])
def test_draws_from_leaf_elements(ctx, orc, R):
    leaf_tiles.test_draws_from_leaf_tiles(ctx, orc, R)
