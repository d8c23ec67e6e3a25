"""The FP64 batched sweep's two ways to sum a Gram (a thread per group and entry, or
a wavefront per group and tile): ranks whose groups do and do not divide a 256-row
chunk, designs and factors of fewer and of more than 32 rows a group, both ways in
one launch and each alone.  Against the oracle's ALS: the nonzeros iterated in the
first sweep are equal and the fits agree to 1e-9, as for the batch's other shapes."""
import numpy as np
import pytest

from conftest import normalized_factors, random_tensor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ranks", [[3], [6], [8, 5], [9, 12, 16], [2, 6, 8, 16, 20]])
@pytest.mark.parametrize("J", [200, 1400, 4000])
def test_batch_gram_routes(ctx, orc, J, ranks):
    from rdist_tensor_amd import abi
    rng = np.random.default_rng(J + len(ranks))
    objs, ref = [], []
    for q, R in enumerate(ranks):
        dims = [700 + q, 40, 33]   # 16 groups at R = 16: more than 32 rows a group in mode 0
        idx, vals = random_tensor(rng, dims, 12000)
        U0 = normalized_factors(rng, dims, R)
        T, F = abi.Tensor(ctx, idx, vals, dims), abi.Factors(ctx, dims, R)
        for k, u in enumerate(U0):
            F.set(k, u)
        S = abi.Sampler(ctx, F, abi.EX_SAMPLER_CP_ARLS_LEV, seed=500 + q)
        A = abi.ALS(ctx, T, F, S)
        A.init()
        objs.append((T, F, S, A))
        ref.append(orc.ALS(idx, vals, dims, U0, "arls", seed=500 + q).run(1, J, 1))
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
