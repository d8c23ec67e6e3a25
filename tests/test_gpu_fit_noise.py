"""The exact fit where |X|^2 + |Xh|^2 - 2 <X, Xh> is negative: rounding noise where
the model reproduces X (fit 1), and a sum that is wrong as a whole where X repeats
coordinates (|X|^2 counts each entry by itself, <X, Xh> their sum): NaN, as the
square root of a negative number is.

Bound of the noise: the terms of each sum have absolute sums of at most (|X| + S)^2,
S = sum_r sigma_r prod_k |u_kr|, and no sum adds more than a few thousand of them
one after another.
"""
import numpy as np
import pytest

from conftest import normalized_factors

pytestmark = pytest.mark.gpu


def fit_of(ctx, idx, vals, dims, U, sigma):
    from rdist_tensor_amd import abi
    T = abi.Tensor(ctx, idx, vals, dims)
    F = abi.Factors(ctx, dims, U[0].shape[1])
    for k, u in enumerate(U):
        F.set(k, u)
    F.set_sigma(sigma)
    A = abi.ALS.exact(ctx, T, F)
    A.init()
    fit = A.fit()
    for x in (A, F, T):
        x.close()
    return fit


@pytest.mark.parametrize("scale", [1.0, 1e-30, 1e30])
def test_repeated_coordinates(ctx, scale):
    dims = [4, 3, 2]
    one = np.indices(dims).reshape(3, -1).T.astype(np.uint32)
    idx = np.concatenate([one, one])
    U = [np.full((d, 1), d ** -0.5) for d in dims]
    # |X|^2 = 48, |Xh|^2 = 96, <X, Xh> = 96 (times scale^2)
    assert np.isnan(fit_of(ctx, idx, np.full(48, scale), dims, U, np.array([2 * scale * 24 ** 0.5])))


@pytest.mark.parametrize("R", [1, 3, 8, 33])
def test_model_reproduces_tensor(ctx, R):
    low = 0
    for seed in range(12):
        rng = np.random.default_rng(100 * R + seed)
        dims = [9, 8, 7]
        U = normalized_factors(rng, dims, R)
        sigma = rng.random(R) + 0.5
        X = np.einsum("ir,jr,kr,r->ijk", *U, sigma)
        idx = np.indices(dims).reshape(3, -1).T.astype(np.uint32)
        vals = X.ravel()
        fit = fit_of(ctx, idx, vals, dims, U, sigma)
        noise = 4097 * np.finfo(float).eps * (np.linalg.norm(vals) + sigma.sum()) ** 2
        assert 1.0 - 1.01 * np.sqrt(noise) / np.linalg.norm(vals) <= fit <= 1.0, (R, seed, fit)
        low += fit == 1.0
    print(f"R {R}: {low} of 12 fits are 1")
