"""The STS-CP draw in each workgroup shape that its rule chooses by rank, samples and
trees: J just below and above one round of small workgroups and of large ones, deep
and shallow trees.  FP64 draws with given uniforms against the oracle: indices exact
except within a boundary's rounding bound (or 1e-12 of it), weights to 1e-11.  Mixed
draws: a sample's draw is keyed by its number, so J changes the shape and not the
draws, and every shape of the same lanes gives the same bits."""
import numpy as np
import pytest

from conftest import normalized_factors

pytestmark = pytest.mark.gpu


def factors(ctx, abi, dims, R):
    rng = np.random.default_rng(R)
    U = [(lambda v: v / np.linalg.norm(v, axis=0))(u + 0.6 / np.sqrt(u.shape[0])) for u in normalized_factors(rng, dims, R)]
    F = abi.Factors(ctx, dims, R)
    for k, u in enumerate(U):
        F.set(k, u)
    return U, F


@pytest.mark.parametrize("dims", [[90, 31, 70], [9000, 31, 400]])
@pytest.mark.parametrize("R", [5, 16, 20, 25, 29, 32, 35, 41, 45])
def test_fp64_shapes_match_oracle(ctx, orc, R, dims):
    from rdist_tensor_amd import abi
    rng = np.random.default_rng(100 + R)
    U, F = factors(ctx, abi, dims, R)
    S = abi.Sampler(ctx, F, abi.EX_SAMPLER_STS_CP, abi.EX_FP64, seed=3)
    so = orc.STS(U)
    for J in ((6144, 6145, 12289, 28000) if R <= 16 else (6145, 8193) if R <= 32 else (3073, 4097)):
        for j in (0, 1):
            de, dr = rng.random((3, J)), rng.random((3, J))
            sg, wg = S.draw(J, j, draws_row=dr, draws_eig=de)
            s_o, wo, margin = so.draw(j, J, de, dr)
            near = (margin < 1e-12) | (so.slack <= 0)
            cols = [k for k in range(3) if k != j]
            moved = np.any(sg[:, cols] != s_o[:, cols], axis=1)
            assert not np.any(moved & ~near), (R, J, j)
            ok = ~moved
            assert np.linalg.norm(wg[ok] - wo[ok]) <= 1e-11 * np.linalg.norm(wo[ok]), (R, J, j)
    S.close()
    F.close()


@pytest.mark.parametrize("dims", [[90, 31, 70], [9000, 31, 400]])
@pytest.mark.parametrize("R", [5, 16, 33, 45, 46, 64])
def test_mixed_shapes_agree(ctx, R, dims):
    from rdist_tensor_amd import abi
    _, F = factors(ctx, abi, dims, R)
    S = abi.Sampler(ctx, F, abi.EX_SAMPLER_STS_CP, abi.EX_MIXED, seed=11)
    for j in (0, 1):
        cols = [k for k in range(3) if k != j]
        many, wm = S.draw(60000, j, sweep=2)
        for J in (700, 6144, 7000, 13000, 28000):
            few, wf = S.draw(J, j, sweep=2)
            assert np.array_equal(many[:J][:, cols], few[:, cols]), (R, J, j)
            assert np.allclose(wm[:J] * (60000 / J), wf, rtol=1e-11), (R, J, j)   # weights carry 1 / J
    S.close()
    F.close()
