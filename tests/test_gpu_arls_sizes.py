"""Leverage scores, their CDF and the column norms of CP-ARLS-LEV at the edges of
the kernels' sizes: ranks around the multiples of 8 that the score kernel is
built for, modes of one row, of a tile of 2048 scores and one more, and of the
four tiles that one workgroup scans and one more; column norms of up to 16 and of
17 blocks of 1024 rows.  Against NumPy in FP64: scores and norms within n
rounding errors of a sum of n terms (1e-12 relative), draws with given uniforms
at the rows of a CDF formed in long double (an index may differ by the CDF's own
rounding only where the uniform lies within 1e-12 of a step)."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R", [1, 8, 9, 33, 64])
def test_scores_cdf_and_norms(ctx, R):
    from rdist_tensor_amd import abi
    dims = [1, 2048, 2049, 8192, 8193, 16385]
    rng = np.random.default_rng(R)
    J = 4000
    for pair in (dims[:3], dims[3:]):
        F = abi.Factors(ctx, pair, R)
        for k, d in enumerate(pair):
            u = rng.standard_normal((d, R)) + 0.1
            F.set(k, u)
            sig = np.empty(R)
            abi.check(abi.lib().ex_factors_renormalize(F.h, k, sig.ctypes.data_as(ctypes.POINTER(ctypes.c_double))))
            want = np.sqrt((u ** 2).sum(0))
            assert np.abs(sig / want - 1).max() < 1e-12
            assert np.abs(F.get(k) * want - u).max() < 1e-12 * np.abs(u).max()
        S = abi.Sampler(ctx, F, abi.EX_SAMPLER_CP_ARLS_LEV, seed=4)
        cdfs = []
        for k, d in enumerate(pair):
            S.update(k)
            u = F.get(k)
            # (fewer rows than columns: the pseudo-inverse is not compared here)
            sc = S.arls_scores(k)
            if d > 4 * R:
                want = np.einsum("ia,ab,ib->i", u, np.linalg.inv(u.T @ u), u)
                assert np.abs(sc - want).max() < 1e-12 * np.abs(want).max()
            c = np.cumsum(sc.astype(np.longdouble))
            cdfs.append((c / c[-1]).astype(np.float64))
        draws = rng.random((len(pair), J))
        for j in range(len(pair)):
            samples, _ = S.draw(J, j, draws_row=draws)
            for k, d in enumerate(pair):
                if k == j or d < 2:
                    continue
                want = np.minimum(np.searchsorted(cdfs[k], draws[k], side="left"), d - 1)
                off = samples[:, k].astype(np.int64) != want
                near = np.abs(cdfs[k][np.minimum(want, samples[:, k])] - draws[k]) < 1e-12
                assert (~off | near).all()
        S.close()
        F.close()
