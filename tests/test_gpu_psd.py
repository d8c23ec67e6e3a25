"""The one-wavefront solves of a positive definite R x R matrix (pinv, the
STS-CP computeM) at the edges of their register layouts (16, 32 and 64
columns; odd orders carry a padding column), and the matrices that they leave
to the two-sided Jacobi: singular, ill conditioned, indefinite, not finite,
eigenvalues at the tolerance or close together.

Tolerances: both sides of a comparison are backward stable solves of an R x R
matrix, so each is within a small multiple of R eps kappa of the exact result
(kappa: largest over smallest kept eigenvalue); 16 R eps kappa covers both.
"""
import numpy as np
import pytest

from conftest import normalized_factors

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps
SIZES = [1, 2, 3, 15, 16, 17, 31, 32, 33, 47, 63, 64]


def spectrum(rng, lam):
    Q, _ = np.linalg.qr(rng.standard_normal((len(lam), len(lam))))
    M = (Q * lam) @ Q.T
    return (M + M.T) / 2


@pytest.mark.parametrize("R", SIZES)
def test_pinv_routes(ctx, orc, R):
    rng = np.random.default_rng(900 + R)
    cases = {
        "well conditioned": rng.uniform(0.5, 2.0, R),
        "graded": np.logspace(0, -6, R) if R > 1 else np.ones(1),
        "scaled up": 1e5 * rng.uniform(0.5, 2.0, R),
        "indefinite": np.where(np.arange(R) % 3 == 1, -1.0, 1.0) * rng.uniform(0.5, 2.0, R),
        "zero": np.zeros(R),
    }
    for name, lam in cases.items():
        M = spectrum(rng, lam)
        kept = np.abs(lam[lam > 1e-11])
        kappa = np.abs(lam).max() / kept.min() if len(kept) else 1.0
        ref, got = orc.pinv(M), ctx.pinv(M)
        assert np.linalg.norm(got - ref) <= 16 * R * EPS * kappa * np.linalg.norm(ref), (R, name)
    # exactly rank-deficient: zero rows, repeated columns
    if R >= 3:
        B = rng.standard_normal((4 * R, R))
        B[:, R // 2] = 0.0
        B[:, R - 1] = B[:, 0]
        M = B.T @ B
        lam = np.linalg.eigvalsh(M)
        kept = lam[lam > 1e-11 * lam.max()]
        ref, got = orc.pinv(M, tol=1e-6), ctx.pinv(M, tol=1e-6)
        assert np.linalg.norm(got - ref) <= 16 * R * EPS * (lam.max() / kept.min()) * np.linalg.norm(ref), R
    # every eigenvalue but the largest below the tolerance
    lam = np.full(R, 1e-4)
    lam[0] = 1.0
    M = spectrum(rng, lam)
    ref, got = orc.pinv(M, tol=1e-3), ctx.pinv(M, tol=1e-3)
    assert np.linalg.norm(got - ref) <= 16 * R * EPS * 1e4 * np.linalg.norm(ref), R


def test_pinv_not_finite(ctx, orc):
    """A NaN or infinite entry: the two-sided solve, entry for entry as the oracle's."""
    for R in (5, 20, 40):
        for bad in (np.nan, np.inf):
            M = np.eye(R)
            M[1, 2] = M[2, 1] = bad
            assert np.array_equal(np.isnan(ctx.pinv(M)), np.isnan(orc.pinv(M))), (R, bad)


@pytest.mark.parametrize("repeat", [False, True])
@pytest.mark.parametrize("R", [1, 2, 15, 17, 32, 33, 64])
def test_compute_m_factorisations(ctx, orc, R, repeat):
    """slot 0 = pinv(H) (1e-8), slot N and slots k the row factors of pinv(H)
    and of (later Grams) (.) pinv(H); rows ordered by eigenvalue, descending in
    slot N and ascending in slots k.  repeat: a repeated column makes H
    singular."""
    from rdist_tensor_amd import abi
    rng = np.random.default_rng(7 * R + repeat)
    for dims in ([90, 70, 80], [70, 90, 66, 75]):
        U = normalized_factors(rng, dims, R)
        if repeat and R > 1:
            for u in U:
                u[:, R - 1] = u[:, 0]
        F = abi.Factors(ctx, dims, R)
        for k, u in enumerate(U):
            F.set(k, u)
        S = abi.Sampler(ctx, F, abi.EX_SAMPLER_STS_CP, abi.EX_FP64, seed=1)
        G = [u.T @ u for u in U]
        N = len(dims)
        for j in range(N):
            M = S.sts_m(j)
            H = np.ones((R, R))
            for k in range(N):
                if k != j:
                    H = H * G[k]
            lam = np.linalg.eigvalsh(H)
            kept = lam[lam > 1e-8]
            tol = 16 * R * EPS * (kept.max() / kept.min())
            P = orc.pinv(H, tol=1e-8)
            assert np.linalg.norm(M[0] - P) <= tol * np.linalg.norm(P), (R, j)
            assert np.linalg.norm(M[N].T @ M[N] - P) <= tol * np.linalg.norm(P), (R, j)
            rows = np.linalg.norm(M[N], axis=1)
            live = rows[rows > 0]
            assert len(live) == len(kept) and np.all(np.diff(live) >= -1e-9 * live.max())
            later = np.ones((R, R))
            for k in range(N - 1, 0, -1):
                if k == j:
                    continue
                later = later * G[k]
                A = later * P
                assert np.linalg.norm(M[k].T @ M[k] - A) <= tol * np.linalg.norm(A), (R, j, k)
                rows = np.linalg.norm(M[k], axis=1)
                assert np.all(np.diff(rows) >= -1e-7 * rows.max()), (R, j, k)
