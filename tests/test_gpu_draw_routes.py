"""The STS-CP draw at the edges of its dispatch: every rank class and vector
count (R), few and many samples, and the first mode's draws from tabulated
masses or by descent.  FP64 draws with injected uniforms against the oracle:
indices exact except within a boundary's rounding bound (or 1e-12 of it),
weights to 1e-11, as for the draws of the other parity tests.  Both routes on
one stream of uniforms: the same draws.
"""
import numpy as np
import pytest

from conftest import normalized_factors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [[900, 31, 400], [40, 700, 300, 65]])
@pytest.mark.parametrize("R", [1, 7, 16, 17, 24, 27, 29, 33, 35, 41, 45, 54, 64])
def test_draws_match_oracle(ctx, orc, R, dims):
    from rdist_tensor_amd import abi
    rng = np.random.default_rng(R)
    U = normalized_factors(rng, dims, R)
    # columns that overlap, so that the Grams are far from the identity
    U = [(lambda v: v / np.linalg.norm(v, axis=0))(u + 0.6 / np.sqrt(u.shape[0])) for u in U]
    F = abi.Factors(ctx, dims, R)
    for k, u in enumerate(U):
        F.set(k, u)
    S = abi.Sampler(ctx, F, abi.EX_SAMPLER_STS_CP, abi.EX_FP64, seed=3)
    so = orc.STS(U)
    N = len(dims)
    for J in (3, 1000, 8200, 30000):
        for j in (0, N - 1):
            de, dr = rng.random((N, J)), rng.random((N, J))
            sg, wg = S.draw(J, j, draws_row=dr, draws_eig=de)
            s_o, wo, margin = so.draw(j, J, de, dr)
            near = (margin < 1e-12) | (so.slack <= 0)
            cols = [k for k in range(N) if k != j]
            moved = np.any(sg[:, cols] != s_o[:, cols], axis=1)
            assert not np.any(moved & ~near), (R, J, j)
            ok = ~moved
            assert np.linalg.norm(wg[ok] - wo[ok]) <= 1e-11 * np.linalg.norm(wo[ok]), (R, J, j)


@pytest.mark.parametrize("R", [8, 16, 32, 64])
def test_routes_agree(ctx, R):
    """The first 8000 draws of 40000 (tabulated first mode) are the 8000-sample
    draw's (descents), which share their uniforms: the sample number keys them."""
    from rdist_tensor_amd import abi
    rng = np.random.default_rng(50 + R)
    dims = [20000, 3000, 700]
    U = normalized_factors(rng, dims, R)
    U = [(lambda v: v / np.linalg.norm(v, axis=0))(u + 0.6 / np.sqrt(u.shape[0])) for u in U]
    F = abi.Factors(ctx, dims, R)
    for k, u in enumerate(U):
        F.set(k, u)
    S = abi.Sampler(ctx, F, abi.EX_SAMPLER_STS_CP, abi.EX_FP64, seed=11)
    for j in range(3):
        many, wm = S.draw(40000, j, sweep=2)
        few, wf = S.draw(8000, j, sweep=2)
        cols = [k for k in range(3) if k != j]
        assert np.array_equal(many[:8000][:, cols], few[:, cols])
        # weights carry 1 / J
        assert np.allclose(wm[:8000] * 5, wf, rtol=1e-11)
