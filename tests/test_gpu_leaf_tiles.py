"""Leaf Grams of the FP64 row trees at the edges of their tiles (2 x 2 up to rank
20, 4 x 4 above, one and three tiles a lane) and with a ragged last leaf: the
factor Gram at the tree's root shapes every draw, so draws with given uniforms are
index-exact against the oracle (draws within 1e-12 of a boundary exempt)."""
import numpy as np
import pytest

from conftest import normalized_factors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R", [2, 5, 20, 21, 33, 63])
def test_draws_from_leaf_tiles(ctx, orc, R):
    from rdist_tensor_amd import abi
    rng = np.random.default_rng(900 + R)
    dims = [400 + R // 2, 3 * R + 1, 97]
    U = normalized_factors(rng, dims, R)
    F = abi.Factors(ctx, dims, R)
    for k in range(3):
        F.set(k, U[k])
    S = abi.Sampler(ctx, F, abi.EX_SAMPLER_STS_CP)
    so = orc.STS(U)
    J = 4000
    for j in range(3):
        de, dr = rng.random((3, J)), rng.random((3, J))
        sg, _ = S.draw(J, j, draws_row=dr, draws_eig=de)
        s_o, _, margin = so.draw(j, J, de, dr)
        near = (margin < 1e-12) | (so.slack <= 0)
        cols = [k for k in range(3) if k != j]
        assert not np.any(np.any(sg[:, cols] != s_o[:, cols], axis=1) & ~near)
    S.close()
    F.close()
