"""The first backward of a mode inside a graph capture, where its key-order copies
of the nonzeros cannot be made: the row-order arrays are gathered instead.  The
scratch of the call is sized by a backward of another mode before it, once
without and once with room for the units of long fibers.

Bound: a gradient entry is a sum of at most n products (n: the nonzeros of the
fibers that meet in it); any order of summation is within 2 (n + 8) eps of the
sum of the absolute terms.
"""
import numpy as np
import pytest

from test_gpu_adjoint_long_fibers import gradients

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R", [3, 16, 64])
@pytest.mark.parametrize("warm", [1, 2])
def test_first_backward_captured(ctx, warm, R):
    import torch
    from rdist_tensor_amd import abi
    from rdist_tensor_amd.autograd import _ptr_array
    rng = np.random.default_rng(90 + R)
    dims = [3000, 2, 3000]
    # long fibers along mode 0 at (b, c) with c < 3, and along mode 2 at (a, b) with a < 3
    parts = []
    for f, n in enumerate([1, 512, 513, 1300, 2500]):
        parts.append(np.stack([3 + rng.choice(dims[0] - 3, n, replace=False), np.full(n, f % 2), np.full(n, f // 2)], 1))
        parts.append(np.stack([np.full(n, f // 2), np.full(n, f % 2), 3 + rng.choice(dims[2] - 3, n, replace=False)], 1))
    idx = np.concatenate(parts).astype(np.uint32)
    vals = rng.standard_normal(len(idx))
    T = abi.Tensor(ctx, idx, vals, dims)
    T.build_lookups()
    U = [torch.as_tensor(rng.standard_normal((d, R))) for d in dims]
    Ud = [u.cuda() for u in U]

    def fibers(mode):
        t = idx.astype(np.int64)
        t[:, mode] = 0
        return np.unique(t, axis=0)

    def backward(stream, mode, sd, w, G, grads):
        abi.check(abi.lib().ex_smttkrp_backward_async(T.h, stream.cuda_stream, mode, len(sd), sd.data_ptr(), w.data_ptr(),
                                                      _ptr_array(Ud), R, G.data_ptr(), _ptr_array(grads)))

    # captured: the long fibers, some short ones, one without nonzeros; before it
    # every fiber of the other mode (more samples, and as many units)
    s0, sw = fibers(0), fibers(warm)
    s0 = np.concatenate([s0[s0[:, 2] < 3], s0[s0[:, 2] >= 3][::7], [[0, 1, 2]]])
    s0 = s0[rng.permutation(len(s0))]
    assert len(sw) > len(s0)
    stream = torch.cuda.Stream()
    d0, dw = (torch.as_tensor(s.astype(np.int32)).cuda() for s in (s0, sw))
    w0 = torch.as_tensor(rng.random(len(s0)) + 0.5)
    G0 = torch.as_tensor(rng.standard_normal((dims[0], R)))
    Gd, wd = G0.cuda(), w0.cuda()
    Gw = torch.ones((dims[warm], R), dtype=torch.float64, device="cuda")
    ww = torch.ones(len(sw), dtype=torch.float64, device="cuda")
    grads = [None, torch.zeros_like(Ud[1]), torch.zeros_like(Ud[2])]
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        backward(stream, warm, dw, ww, Gw, [torch.zeros_like(u) if k != warm else None for k, u in enumerate(Ud)])
    stream.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        for g in grads[1:]:
            g.zero_()
        backward(stream, 0, d0, wd, Gd, grads)
    where = {tuple(t[1:]): c for c, t in enumerate(s0.tolist())}
    hit = np.array([(int(b), int(c)) in where for _, b, c in idx.tolist()])
    cs = torch.as_tensor([where[(int(b), int(c))] for _, b, c in idx[hit].tolist()])
    rows, xs, sdt = torch.as_tensor(idx[hit, 0].astype(np.int64)), torch.as_tensor(vals[hit]), torch.as_tensor(s0)
    ref = gradients(torch, rows, cs, xs, sdt, w0, U, G0, R)
    mag = gradients(torch, rows, cs, xs.abs(), sdt, w0, [u.abs() for u in U], G0.abs(), R)
    bound = 2 * (len(idx) + 8) * np.finfo(np.float64).eps

    def check(got, what):
        for k in range(2):
            assert bool(((got[k + 1].cpu() - ref[k]).abs() <= bound * mag[k]).all()), (what, warm, R, k)

    for replay in range(3):
        Gd.mul_(1.0)   # the program's own eager work between the replays
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        check(grads, replay)
    # eager afterwards: the copies are made now
    eager = [None, torch.zeros_like(Ud[1]), torch.zeros_like(Ud[2])]
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        backward(stream, 0, d0, wd, Gd, eager)
    torch.cuda.synchronize()
    check(eager, "eager")
    graph.replay()
    torch.cuda.synchronize()
    check(grads, "after")
