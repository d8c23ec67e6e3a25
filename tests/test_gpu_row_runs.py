"""Row sums run by run (the sampled and the exact MTTKRP's pass over the
nonzeros): ranks that do and do not fill the lanes of a run or the 64 lanes of a
wavefront, tensors of one nonzero, of one chunk of 256 and of one more or less,
rows that end inside a run, between runs and chunks, and that span several chunks.
FP64 sampled sums against the sums formed in long double (1e-12 relative: at most
2000 terms a row), exact ALS steps against the oracle (FP64 1e-9; mixed 1e-5: FP32
sums, well-conditioned Grams)."""
import numpy as np
import pytest

from conftest import normalized_factors
from test_gpu_exact import skewed_tensor

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(np.asarray(a, float) - np.asarray(b, float)) / max(np.linalg.norm(np.asarray(b, float)), 1e-300)


@pytest.mark.parametrize("R", [1, 2, 3, 7, 20, 33, 63, 64])
def test_sampled_rows(ctx, R):
    from rdist_tensor_amd import abi
    rng = np.random.default_rng(R)
    dims = [700, 90, 80]
    for nnz in (1, 255, 256, 257, 6000):
        idx, vals = skewed_tensor(rng, dims, nnz)
        T = abi.Tensor(ctx, idx, vals, dims)
        T.mttkrp_path(1)   # the row pass
        T.build_lookups()
        for share in (1.0, 0.1):
            fib, inv = np.unique(idx[:, 1].astype(np.int64) * dims[2] + idx[:, 2], return_inverse=True)
            keep = rng.random(len(fib)) < share
            keep[0] = True
            sd = np.zeros((keep.sum(), 3), np.uint32)
            sd[:, 1], sd[:, 2] = fib[keep] // dims[2], fib[keep] % dims[2]
            D = rng.standard_normal((len(sd), R))
            at = np.cumsum(keep) - 1
            hit = keep[inv]
            want = np.zeros((dims[0], R), np.longdouble)
            np.add.at(want, idx[hit, 0], vals[hit, None].astype(np.longdouble) * D[at[inv[hit]]])
            Y, H = T.sampled_mttkrp(0, sd, D)
            assert H == hit.sum()
            assert rel(Y, want) < 1e-12
        T.close()


@pytest.mark.parametrize("precision,bar", [("fp64", 1e-9), ("mixed", 1e-5)])
@pytest.mark.parametrize("R", [1, 3, 5, 20, 33])
def test_exact_steps(ctx, orc, R, precision, bar):
    from rdist_tensor_amd import abi
    rng = np.random.default_rng(100 + R)
    dims = [900, 300, 250]
    idx, vals = skewed_tensor(rng, dims, 20000)
    U = normalized_factors(rng, dims, R)
    T, F = abi.Tensor(ctx, idx, vals, dims), abi.Factors(ctx, dims, R)
    for k, u in enumerate(U):
        F.set(k, u)
    A = abi.ALS.exact(ctx, T, F, precision=abi.EX_MIXED if precision == "mixed" else abi.EX_FP64)
    A.init()
    for j in range(3):
        oa = orc.ALS(idx, vals, dims, U, "exact")
        oa.step(j, 0, 1)
        A.step(j, 0, 1)
        err = rel(F.get(j), oa.U[j])
        print(f"{precision} R={R} mode {j}: {err:.2e}")
        assert err < bar
        U[j] = F.get(j)   # the next step's Grams and rows are this side's
    for x in (A, F, T):
        x.close()
