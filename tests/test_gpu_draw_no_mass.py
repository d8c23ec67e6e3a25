"""Mixed STS-CP draws where the first drawn mode has no mass (its factor is zero):
every component's table is flat, so no entry passes the target.  65 tiles of 32
leaves: more than the lanes of a group, with pieces that fewer lanes cover.  Every
sample stays inside its mode, with weight 0."""
import numpy as np
import pytest

from conftest import normalized_factors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,knob", [(16, None), (16, ("sts_draw.fp32.r16", 0)), (32, None), (40, None), (64, None),
                                    (64, ("sts_draw.fp32.r64", 0))])
def test_samples_stay_in_range(ctx, R, knob):
    from rdist_tensor_amd import abi
    dims = [64 * 32 * R + 5, 300, 200]   # a leaf holds R rows
    U = normalized_factors(np.random.default_rng(3), dims, R)
    U[0][:] = 0.0
    before = abi.tuning()
    if knob:
        abi.tuning_set(*knob)
    try:
        F = abi.Factors(ctx, dims, R)
        for k in range(3):
            F.set(k, U[k])
        S = abi.Sampler(ctx, F, abi.EX_SAMPLER_STS_CP, precision=abi.EX_MIXED, seed=9)
        for j in (1, 2):
            samples, w = S.draw(5000, j, sweep=2)
            for k in (0, 3 - j):
                assert samples[:, k].max() < dims[k]
            assert np.all(w == 0.0)
    finally:
        if knob:
            abi.tuning_set(knob[0], before[knob[0]][1])
