"""The FP64 batched sweep at the edges of its dispatch (kernels_batch64.hip):
ranks whose Gram groups do and do not divide a 256-row chunk, one and three Gram
tiles, sample counts that leave partial workgroups, three and four modes in one
batch.  Against the oracle's ALS: the nonzeros iterated in the first sweep are
equal (the same draws and the same fibers) and the fits agree to 1e-9."""
import numpy as np
import pytest

from conftest import normalized_factors, random_tensor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("J", [255, 1025, 8192])
def test_batch_ranks_and_modes(ctx, orc, J):
    from rdist_tensor_amd import abi
    rng = np.random.default_rng(J)
    objs, ref = [], []
    for q, R in enumerate([1, 2, 3, 4, 7, 10, 16, 17, 31, 32]):
        if J < 8 * R:
            continue
        dims = [50 + q, 40, 33] if q % 3 else [14, 13 + q, 12, 11]
        idx, vals = random_tensor(rng, dims, 12000)
        U0 = normalized_factors(rng, dims, R)
        T, F = abi.Tensor(ctx, idx, vals, dims), abi.Factors(ctx, dims, R)
        for k, u in enumerate(U0):
            F.set(k, u)
        S = abi.Sampler(ctx, F, abi.EX_SAMPLER_CP_ARLS_LEV, seed=300 + q)
        A = abi.ALS(ctx, T, F, S)
        A.init()
        objs.append((T, F, S, A))
        ref.append(orc.ALS(idx, vals, dims, U0, "arls", seed=300 + q).run(1, J, 1))
    B = abi.Batch([o[3] for o in objs], J)
    B.run(1)
    nz = B.counters()[0]
    for o, n, (fits, st) in zip(objs, nz, ref):
        assert n == st["nonzeros_iterated"]
        assert abs(o[3].fit() - fits[-1]) < 1e-9
    B.close()
    for o in objs:
        for x in reversed(o):
            x.close()
