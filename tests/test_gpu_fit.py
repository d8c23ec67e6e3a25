"""The exact fit at the edges of its kernel (chunks of 256 nonzeros, two columns
per lane, every lane layout, each choice of the row order) against the oracle.

Bound: |X|^2, |Xh|^2 and <X, Xh> are sums of at most nnz, R^2 and nnz R products;
each order of summation is within (terms) eps of the absolute sum, and the fit
1 - sqrt(res2) / |X| moves by half the error of res2 over sqrt(res2) |X|.
"""
import numpy as np
import pytest

from conftest import normalized_factors, random_tensor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [[40, 30], [30, 41, 23], [23, 30, 41], [9, 8, 7, 11], [700, 5, 600]])
@pytest.mark.parametrize("R", [1, 3, 8, 16, 25, 32, 33, 64])
def test_fit(ctx, orc, R, dims):
    from rdist_tensor_amd import abi
    for nnz in (1, 255, 256, 257, 1200):
        rng = np.random.default_rng(R * 1000 + nnz)
        idx, vals = random_tensor(rng, dims, min(nnz, int(np.prod(dims)) // 2))
        U = normalized_factors(rng, dims, R)
        T = abi.Tensor(ctx, idx, vals, dims)
        F = abi.Factors(ctx, dims, R)
        for k, u in enumerate(U):
            F.set(k, u)
        A = abi.ALS.exact(ctx, T, F)
        A.init()
        ref = orc.ALS(idx, vals, dims, U, "exact").fit()
        terms = np.abs(vals) * np.prod([np.abs(U[k])[idx[:, k]] for k in range(len(dims))], axis=0).sum(1)
        had = np.prod([np.abs(u).T @ np.abs(u) for u in U], axis=0).sum()
        size = (vals ** 2).sum() + had + 2 * terms.sum()
        norm = np.linalg.norm(vals)
        res = max((1 - ref) * norm, 1e-300)
        n = len(idx) * (R + len(dims)) + R * R + sum(dims)
        assert abs(A.fit() - ref) <= 2 * n * np.finfo(float).eps * size / (res * norm), (R, dims, nnz)
