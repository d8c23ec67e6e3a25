"""The mixed sampled MTTKRP's row sums run by run, at ranks that do and do not fill
the lanes of a run, both lane counts: one mode step from known factors.  Its update
is U_j diag(sigma) = Y A with one R x R matrix A for all rows (the pseudo-inverse of
a BF16 Gram), so with Y summed here in FP64 from the step's own draws, A found by
least squares leaves a residual of FP32 rounding only; a row that misses a hit, a
column or a run leaves much more.

Bound: row i's sum of n_i products of N FP32 rows and a weight is within (n_i + 2 N +
4) eps of its absolute sum Yabs_i, its product with A within (R + 4) eps of Yabs_i |A|
more; A's own error is of the same kind, hence twice that.

And the mixed computeM at ranks that do not divide its 1024 threads."""
import numpy as np
import pytest

import test_gpu_mixed as mixed
from conftest import normalized_factors
from test_gpu_exact import skewed_tensor
from test_gpu_tuning import knob  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("R", [1, 3, 5, 20, 33, 63, 64])
def test_mixed_sampled_rows(ctx, knob, R, variant):  # noqa: F811
    from rdist_tensor_amd import abi
    knob("row_scan.fp32", variant)
    rng = np.random.default_rng(R)
    dims = [700, 90, 80]
    idx, vals = skewed_tensor(rng, dims, 30000)
    vals = vals.astype(np.float32).astype(np.float64)   # exact in the pass's copy
    U = [u.astype(np.float32).astype(np.float64) for u in normalized_factors(rng, dims, R)]
    T, F = abi.Tensor(ctx, idx, vals, dims), abi.Factors(ctx, dims, R)
    T.mttkrp_path(abi.EX_MTTKRP_ROW_PASS)
    for k, u in enumerate(U):
        F.set(k, u)
    S = abi.Sampler(ctx, F, abi.EX_SAMPLER_CP_ARLS_LEV, precision=abi.EX_MIXED, seed=9)
    A = abi.ALS(ctx, T, F, S, precision=abi.EX_MIXED)
    A.init()
    J = 6000
    s, w = S.draw(J, 0, sweep=1)
    key, first, mult = np.unique(s[:, 1].astype(np.int64) * dims[2] + s[:, 2], return_index=True, return_counts=True)
    D = U[1][s[first, 1]] * U[2][s[first, 2]] * (w[first] * mult)[:, None]
    nz = idx[:, 1].astype(np.int64) * dims[2] + idx[:, 2]
    at = np.minimum(np.searchsorted(key, nz), len(key) - 1)
    hit = key[at] == nz
    Y, Yabs, n = np.zeros((dims[0], R)), np.zeros((dims[0], R)), np.zeros(dims[0])
    np.add.at(Y, idx[hit, 0], vals[hit, None] * D[at[hit]])
    np.add.at(Yabs, idx[hit, 0], np.abs(vals[hit, None] * D[at[hit]]))
    np.add.at(n, idx[hit, 0], 1)
    A.step(0, J, 1)
    got = F.get(0) * F.sigma()
    assert (n > 0).sum() > 4 * R and not got[n == 0].any()
    M = np.linalg.lstsq(Y, got, rcond=None)[0]
    eps = np.finfo(np.float32).eps
    bound = 2 * eps * (n[:, None] + R + 2 * 3 + 8) * (Yabs @ np.abs(M))
    worst = np.max(np.abs(Y @ M - got)[n > 0] / bound[n > 0])
    print(f"R={R} variant {variant}: {int(hit.sum())} hits, residual up to {worst:.2g} of its bound")
    assert worst <= 1
    for x in (A, S, F, T):
        x.close()


@pytest.mark.parametrize("R", [33, 45, 63])
def test_mixed_compute_m_ranks(ctx, R):
    mixed.test_mixed_compute_m_factorisations(ctx, R)
