"""The adjoint of the sampled MTTKRP where fibers are longer than one unit of
its kernels (512 nonzeros): lengths around one and several units, every lane
layout of a gradient row, and an output gradient that is not 16-byte aligned.

Bound: a gradient entry is a sum of at most n products (n: the nonzeros of the
fibers that meet in it); any order of summation is within 2 (n + 8) eps of the
sum of the absolute terms.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LENGTHS = [1, 2, 511, 512, 513, 1023, 1024, 1025, 5000]


def gradients(torch, rows, cs, xs, sd, wd, U, G, ncol):
    """dL/dU_1 and dL/dU_2 for mode 0 of a 3-mode tensor, in FP64 on the CPU."""
    u1, u2 = U[1][sd[:, 1]], U[2][sd[:, 2]]
    dD = torch.zeros(len(sd), ncol, dtype=torch.float64).index_add_(0, cs, xs[:, None] * G[rows]) * wd[:, None]
    g1 = torch.zeros_like(U[1]).index_add_(0, sd[:, 1], dD * u2)
    g2 = torch.zeros_like(U[2]).index_add_(0, sd[:, 2], dD * u1)
    return g1, g2


@pytest.mark.parametrize("R", [1, 3, 8, 16, 25, 32, 33, 64])
def test_long_fibers(ctx, R):
    import torch
    from rdist_tensor_amd import abi
    from rdist_tensor_amd.autograd import SampledMTTKRP
    rng = np.random.default_rng(40 + R)
    dims = [6000, 3, 4]
    idx = []
    for f, n in enumerate(LENGTHS):
        rows = rng.choice(dims[0], size=n, replace=False)
        idx.append(np.stack([rows, np.full(n, f % 3), np.full(n, f // 3)], 1))
    idx = np.concatenate(idx).astype(np.uint32)
    vals = rng.standard_normal(len(idx))
    T = abi.Tensor(ctx, idx, vals, dims)
    T.build_lookups()
    # every fiber sampled, and one tuple without nonzeros
    sd = np.array([[0, f % 3, f // 3] for f in range(len(LENGTHS))] + [[0, 2, 3]])
    order = rng.permutation(len(sd))
    sd = sd[order]
    where = {tuple(t[1:]): c for c, t in enumerate(sd.tolist())}
    cs = torch.as_tensor([where[(int(b), int(c))] for _, b, c in idx.tolist()])
    wd = torch.as_tensor(rng.random(len(sd)) + 0.5)
    U = [torch.as_tensor(rng.standard_normal((d, R))) for d in dims]
    G = torch.as_tensor(rng.standard_normal((dims[0], R)))
    sdt, rows, xs = torch.as_tensor(sd), torch.as_tensor(idx[:, 0].astype(np.int64)), torch.as_tensor(vals)
    ref = gradients(torch, rows, cs, xs, sdt, wd, U, G, R)
    mag = gradients(torch, rows, cs, xs.abs(), sdt, wd, [u.abs() for u in U], G.abs(), R)
    bound = 2 * (sum(LENGTHS) + 8) * np.finfo(np.float64).eps
    samples = torch.as_tensor(sd.astype(np.int32)).cuda()
    for aligned in (True, False):
        if aligned:
            Gd = G.cuda()
        else:
            Gd = torch.empty(G.numel() + 1, dtype=torch.float64, device="cuda")[1:].view(G.shape)
            Gd.copy_(G)
        for _ in range(2):   # the unit lists are cleared by each call
            Ud = [u.cuda().requires_grad_(k > 0) for k, u in enumerate(U)]
            Y = SampledMTTKRP.apply(T, 0, samples, wd.cuda(), *Ud)
            got = torch.autograd.grad(Y, Ud[1:], Gd)
            for k in range(2):
                assert bool(((got[k].cpu() - ref[k]).abs() <= bound * mag[k]).all()), (R, aligned, k)


def test_repeated_samples_with_long_fibers(ctx):
    """Repeated tuples on long fibers: every gradient NaN, and a call after it is whole again."""
    import torch
    from rdist_tensor_amd import abi
    from rdist_tensor_amd.autograd import SampledMTTKRP
    rng = np.random.default_rng(3)
    dims, R, n = [3000, 2, 2], 8, 2500
    idx = np.concatenate([np.stack([rng.choice(dims[0], n, replace=False), np.full(n, a), np.full(n, b)], 1)
                          for a in range(2) for b in range(2)]).astype(np.uint32)
    T = abi.Tensor(ctx, idx, rng.standard_normal(len(idx)), dims)
    T.build_lookups()
    U = [torch.as_tensor(rng.standard_normal((d, R))).cuda() for d in dims]
    G = torch.as_tensor(rng.standard_normal((dims[0], R))).cuda()

    def grads(s):
        Ud = [u.clone().requires_grad_(k > 0) for k, u in enumerate(U)]
        s = torch.as_tensor(np.array(s, np.int32)).cuda()
        w = torch.ones(len(s), dtype=torch.float64, device="cuda")
        return torch.autograd.grad(SampledMTTKRP.apply(T, 0, s, w, *Ud), Ud[1:], G)

    good = [[0, 0, 0], [0, 1, 0], [0, 0, 1], [0, 1, 1]]
    before = grads(good)
    for g in grads([[0, 0, 1]] * 200 + good):
        assert bool(torch.isnan(g).all())
    for a, b in zip(before, grads(good)):
        assert float((a - b).abs().max()) <= 1e-12 * float(a.abs().max())
