"""One optimizer stepped with sample counts that grow: the deduplication's table is
replaced by a larger one each time, possibly at the address of the one freed for it,
and must start empty.  Every step equals that of a fresh optimizer, bit for bit."""
import numpy as np
import pytest

from conftest import normalized_factors, random_tensor

pytestmark = pytest.mark.gpu


def test_steps_with_growing_tables(ctx):
    from rdist_tensor_amd import abi
    rng = np.random.default_rng(7)
    dims, R = [300, 200, 100], 8
    idx, vals = random_tensor(rng, dims, 20000)
    T = abi.Tensor(ctx, idx, vals, dims)
    T.build_lookups()
    U = normalized_factors(rng, dims, R)

    def optimizer():
        F = abi.Factors(ctx, dims, R)
        for k in range(3):
            F.set(k, U[k])
        S = abi.Sampler(ctx, F, abi.EX_SAMPLER_CP_ARLS_LEV, seed=5)
        A = abi.ALS(ctx, T, F, S)
        A.init()
        return A, S, F

    A, S, F = optimizer()
    for n, J in enumerate([300, 900, 5000, 40, 33000, 70000, 300]):
        F.set(0, U[0])
        S.update(0)
        A.step(0, J, 1 + n)
        B, SB, FB = optimizer()
        B.step(0, J, 1 + n)
        assert np.array_equal(F.get(0), FB.get(0))
        for x in (B, SB, FB):
            x.close()
