"""The adjoint of the sampled MTTKRP at short fibers: one nonzero, and lengths
around the number S of nonzeros that a wavefront takes side by side (1 to 32 by the
rank) and around a batch of four times as many.

Bound: a gradient entry is a sum of at most n products (n: the nonzeros of the
fibers that meet in it); any order of summation is within 2 (n + 8) eps of the
sum of the absolute terms.
"""
import numpy as np
import pytest

from test_gpu_adjoint_long_fibers import gradients

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R", [1, 4, 5, 8, 16, 21, 32, 33, 64])
def test_short_fibers(ctx, R):
    import torch
    from rdist_tensor_amd import abi
    from rdist_tensor_amd.autograd import SampledMTTKRP
    rng = np.random.default_rng(60 + R)
    lanes = 2
    while lanes < (R + 1) // 2:
        lanes *= 2
    S = 64 // lanes
    lengths = sorted({1, 2, 3, S - 1, S, S + 1, 2 * S, 4 * S, 4 * S + 1} - {0}) * 2
    dims = [200, 5, 5]
    idx = np.concatenate([np.stack([rng.choice(dims[0], n, replace=False), np.full(n, f % 5), np.full(n, f // 5)], 1)
                          for f, n in enumerate(lengths)]).astype(np.uint32)
    vals = rng.standard_normal(len(idx))
    T = abi.Tensor(ctx, idx, vals, dims)
    T.build_lookups()
    sd = rng.permutation(np.array([[0, f % 5, f // 5] for f in range(len(lengths))] + [[0, 4, 4]]))
    where = {tuple(t[1:]): c for c, t in enumerate(sd.tolist())}
    cs = torch.as_tensor([where[(int(b), int(c))] for _, b, c in idx.tolist()])
    wd = torch.as_tensor(rng.random(len(sd)) + 0.5)
    U = [torch.as_tensor(rng.standard_normal((d, R))) for d in dims]
    G = torch.as_tensor(rng.standard_normal((dims[0], R)))
    sdt, rows, xs = torch.as_tensor(sd), torch.as_tensor(idx[:, 0].astype(np.int64)), torch.as_tensor(vals)
    ref = gradients(torch, rows, cs, xs, sdt, wd, U, G, R)
    mag = gradients(torch, rows, cs, xs.abs(), sdt, wd, [u.abs() for u in U], G.abs(), R)
    bound = 2 * (sum(lengths) + 8) * np.finfo(np.float64).eps
    Ud = [u.cuda().requires_grad_(k > 0) for k, u in enumerate(U)]
    Y = SampledMTTKRP.apply(T, 0, torch.as_tensor(sd.astype(np.int32)).cuda(), wd.cuda(), *Ud)
    got = torch.autograd.grad(Y, Ud[1:], G.cuda())
    for k in range(2):
        assert bool(((got[k].cpu() - ref[k]).abs() <= bound * mag[k]).all()), (R, k)
