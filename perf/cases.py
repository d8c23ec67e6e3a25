"""The work that a program using rdist_tensor_amd has it do, as cases to time.

A case is a dict of plain values.  `kind` is the call that a program makes:

* ``run``     a whole decomposition call: initial factors set, the sampler
              built from them, `sweeps` sweeps of the randomized optimizer
              with the exact fit at the end, the factors read back;
* ``step``    one mode step of the randomized optimizer (draw, deduplicate,
              design and its pseudo-inverse, sampled MTTKRP, factor update,
              sampler update) from the factors of a decomposition under way,
              the updated factor read back;
* ``exact``   sweeps of the non-randomized optimizer (every nonzero);
* ``batch``   sweeps of many small CP-ARLS-LEV decompositions in one launch each;
* ``adjoint`` the differentiable sampled MTTKRP, forward and backward, on
              torch tensors that stay on the GPU.

FP64 is the reference's arithmetic and the default; mixed precision holds the
factors in FP32, and a program on that path keeps them as such.  Mixed cases
are single steps, or sweeps without draws: each draws its samples from the
factors of the step before.

Sizes are those of the benchmark configurations (rdist_tensor_amd/synthetic.py)
and of the tests, at full size or scaled; Zipf exponents, ranks, sample counts
and value distributions likewise.
"""
import ctypes
import json
import math

import numpy as np
import torch

from rdist_tensor_amd import abi, autograd

_CTX = []


def _context():
    if not _CTX:
        torch.cuda.init()
        _CTX.append(abi.Context(0))
    return _CTX[0]


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest decompositions (the tests' sizes): every kernel is short,
        # launches and the R x R solves count
        dict(name="run arls 300x200x100 R8", kind="run", sampler="arls", precision="fp64", dims="300,200,100",
             nnz=30_000, zipf="", values="uniform", R=8, J=1000, sweeps=5, graph=False),
        # the reference's own CPU-sized problem, replayed from a graph
        dict(name="run arls 2000^3 R16", kind="run", sampler="arls", precision="fp64", dims="2000,2000,2000",
             nnz=200_000, zipf="1.1,1.1,1.1", values="uniform", R=16, J=32768, sweeps=10, graph=True),
        # the same problem on the mixed path, one mode
        dict(name="step arls 2000^3 R16 mixed", kind="step", sampler="arls", precision="mixed",
             dims="2000,2000,2000", nnz=200_000, zipf="1.1,1.1,1.1", values="uniform", R=16, J=32768, mode=1),
        # four modes, the exact Khatri-Rao sampler, a size where its R x R
        # work outweighs the passes over the tensor
        dict(name="run sts 4 modes R16", kind="run", sampler="sts", precision="fp64", dims="70,60,50,31",
             nnz=200_000, zipf="", values="uniform", R=16, J=8192, sweeps=3, graph=False),
        # an ordinary FROSTT-sized tensor at the reference's usual rank of 25
        # (odd: no vector width divides it), ragged modes
        dict(name="run sts 2e6 nnz R25", kind="run", sampler="sts", precision="fp64", dims="60013,40001,9001",
             nnz=2_000_000, zipf="1.1,1.1,1.1", values="lognormal", R=25, J=65536, sweeps=2, graph=False),
        # a large tensor in the reference's arithmetic
        dict(name="run sts 2e7 nnz R32", kind="run", sampler="sts", precision="fp64", dims="500000,300000,50000",
             nnz=20_000_000, zipf="1.1,1.1,1.1", values="lognormal", R=32, J=65536, sweeps=3, graph=False),
        # the benchmark's tensor on the mixed path: draws over both million-row modes
        dict(name="step sts 5e7 nnz R32 mixed", kind="step", sampler="sts", precision="mixed",
             dims="1000000,1000000,100000", nnz=50_000_000, zipf="1.1,1.1,1.1", values="lognormal", R=32, J=65536,
             mode=2),
        # four modes at the largest rank, mixed path
        dict(name="step sts 4 modes R64 mixed", kind="step", sampler="sts", precision="mixed",
             dims="1000000,200000,10000,100", nnz=20_000_000, zipf="1.2,1.2,0,0", values="poisson", R=64, J=131072,
             mode=2),
        # exact ALS, the reference's non-randomized optimizer
        dict(name="exact 3e6 nnz R32", kind="exact", precision="fp64", dims="50000,30000,8000", nnz=3_000_000,
             zipf="1.1,1.1,1.1", values="lognormal", R=32, sweeps=2),
        # exact ALS on the mixed path at a rank that is no multiple of 16
        dict(name="exact 1e7 nnz R20 mixed", kind="exact", precision="mixed", dims="100003,80001,20011",
             nnz=10_000_000, zipf="1.1,1.1,1.1", values="lognormal", R=20, sweeps=1),
        # many small decompositions at once
        dict(name="batch of 32, R8-32", kind="batch", precision="fp64", count=32, low=60, high=600, J=8192, sweeps=5),
        # first-order fitting: sampled MTTKRP and its adjoint at the benchmark's size
        dict(name="adjoint 2e7 nnz R32", kind="adjoint", precision="fp64", dims="500000,500000,500000",
             nnz=20_000_000, zipf="1.1,1.1,1.1", values="lognormal", R=32, J=65536, mode=0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["run", "run", "run", "step", "step", "exact", "batch", "adjoint"])
    if kind == "batch":
        low = _log_int(rng, 40, 120)
        return dict(kind="batch", precision="fp64", count=rng.randint(4, 40), low=low, high=_log_int(rng, 300, 900),
                    J=_log_int(rng, 1000, 8192), sweeps=rng.randint(1, 6))
    N = 4 if rng.random() < 0.25 else 3
    nnz = _log_int(rng, 5_000, 10_000_000)
    # modes between a handful of rows and about the nonzeros' number; the
    # nonzeros fill at most a twentieth of the tensor
    dims = []
    for k in range(N):
        dims.append(_log_int(rng, 60 if N == 3 else 30, max(200, min(400_000, nnz // 10))))
    while math.prod(dims) < 20 * nnz:
        k = rng.randrange(N)
        dims[k] = int(dims[k] * 1.5) + 1
    # skewed like the benchmark's tensor, or uniform: a randomized optimizer's
    # samples then only find nonzeros where the tensor is not too sparse
    zipf = ",".join("1.1" for _ in dims) if rng.random() < 0.5 else ""
    if not zipf and kind in ("run", "step"):
        while math.prod(dims) > 300 * nnz:
            dims[dims.index(max(dims))] = max(dims) * 2 // 3
    while zipf and math.prod(dims) > 1_000_000 * nnz:
        dims[dims.index(max(dims))] = max(dims) * 2 // 3
    while zipf and math.prod(dims) < 1000 * nnz:
        k = rng.randrange(N)
        dims[k] = int(dims[k] * 1.5) + 1
    base = dict(dims=",".join(map(str, dims)), nnz=nnz, zipf=zipf,
                values=rng.choice(["uniform", "lognormal", "poisson"]))
    if kind == "exact":
        return dict(kind=kind, precision=rng.choice(["fp64", "mixed"]), R=rng.randint(3, 40),
                    sweeps=rng.randint(1, 2) if nnz < 2_000_000 else 1, **base)
    J = _log_int(rng, 1000, 100_000)
    if kind == "adjoint":
        return dict(kind=kind, precision="fp64", R=rng.randint(3, 64), J=J, mode=rng.randrange(N), **base)
    sampler = rng.choice(["arls", "sts"])
    R = rng.choice([rng.randint(4, 16), rng.randint(17, 32), rng.randint(33, 64)])
    J = max(J, 200 * R)   # a least-squares problem needs many samples per unknown
    if kind == "step":
        return dict(kind=kind, sampler=sampler, precision="mixed", R=R, J=J, mode=dims.index(min(dims)), **base)
    return dict(kind=kind, sampler=sampler, precision="fp64", R=R, J=J, sweeps=rng.randint(1, 3) if R <= 32 else 1,
                graph=rng.random() < 0.5, **base)


def _dims(case):
    return [int(d) for d in case["dims"].split(",")]


# ---------------------------------------------------------------- inputs
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1_000_003 + 17)
    return g


def _coordinates(g, dims, nnz, zipf):
    """`nnz` distinct coordinates (int64, nnz x N), in random order: uniform, or
    per mode Zipf over randomly permuted ranks."""
    exponents = [float(z) for z in zipf.split(",")] if zipf else [0.0] * len(dims)
    cdfs = []
    for d, z in zip(dims, exponents):
        if z:
            p = torch.arange(1, d + 1, device="cuda", dtype=torch.float64) ** -z
            c = torch.cumsum(p, 0)
            cdfs.append((c / c[-1], torch.randperm(d, generator=g, device="cuda")))
        else:
            cdfs.append(None)
    have = torch.empty(0, dtype=torch.int64, device="cuda")
    while have.numel() < nnz:
        n = int((nnz - have.numel()) * 1.2) + 1024
        lin = torch.zeros(n, dtype=torch.int64, device="cuda")
        for d, c in zip(dims, cdfs):
            if c is None:
                i = torch.randint(d, (n,), generator=g, device="cuda")
            else:
                u = torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
                i = c[1][torch.searchsorted(c[0], u).clamp_(max=d - 1)]
            lin = lin * d + i
        have = torch.unique(torch.cat([have, lin]))
    lin = have[torch.randperm(have.numel(), generator=g, device="cuda")[:nnz]]
    out = torch.empty((nnz, len(dims)), dtype=torch.int64, device="cuda")
    for k in range(len(dims) - 1, -1, -1):
        out[:, k] = lin % dims[k]
        lin = lin // dims[k]
    return out


def _values(g, n, kind):
    if kind == "uniform":
        return torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    if kind == "lognormal":
        return torch.randn(n, generator=g, device="cuda", dtype=torch.float64).exp().float().double()
    rate = torch.full((n,), 2.0, device="cuda", dtype=torch.float64)
    return 1.0 + torch.poisson(rate, generator=g)


def _factors(g, dims, R):
    """N(0,1) factors with unit columns, as the library's users start from."""
    U = [torch.randn((d, R), generator=g, device="cuda", dtype=torch.float64) for d in dims]
    return [u / u.norm(dim=0) for u in U]


def _factors_under_way(g, dims, R, coords):
    """Factors some sweeps into a decomposition: a row's norm follows its share
    of the nonzeros, so the leverage samples fall on the fibers that hold them."""
    U = _factors(g, dims, R)
    for k, u in enumerate(U):
        share = torch.bincount(coords[:, k], minlength=dims[k]).double()
        u *= share.sqrt()[:, None]
        u /= u.norm(dim=0)
    return U


def _host(u):
    """A pinned host copy: what a program hands to the library and reads into."""
    h = torch.empty(u.shape, dtype=u.dtype, pin_memory=True)
    h.copy_(u)
    return h


def _raw(case, seed):
    g = _generator(seed)
    dims = _dims(case)
    coords = _coordinates(g, dims, case["nnz"], case["zipf"])
    vals = _values(g, case["nnz"], case["values"])
    return g, dims, coords, vals


def _precision(case):
    return abi.EX_MIXED if case["precision"] == "mixed" else abi.EX_FP64


def _sampler(ctx, case, F, seed):
    kind = abi.EX_SAMPLER_STS_CP if case["sampler"] == "sts" else abi.EX_SAMPLER_CP_ARLS_LEV
    return abi.Sampler(ctx, F, kind, _precision(case), seed=seed)


def _tensor(ctx, dims, coords, vals):
    return abi.Tensor(ctx, coords.to(torch.int32).cpu().numpy().view(np.uint32), vals.cpu().numpy(), dims)


def _batch_tensors(case, seed):
    """Sizes, ranks and nonzeros of each tensor of a batch: the nonzeros fill
    a quarter of the longest mode's fibers many times over."""
    import random
    r = random.Random(seed)
    shapes = random.Random(case["count"] * 1009 + case["low"])
    out = []
    for _ in range(case["count"]):
        dims = [shapes.randint(case["low"], case["high"]) for _ in range(3)]
        out.append((dims, min(60 * max(dims), math.prod(dims) // 20), shapes.choice([8, 16, 32]), r.randrange(1 << 30)))
    return out


def prepare(case, seed):
    ctx = _context()
    if case["kind"] == "batch":
        members = []
        for dims, nnz, R, s in _batch_tensors(case, seed):
            g = _generator(s)
            T = _tensor(ctx, dims, _coordinates(g, dims, nnz, ""), _values(g, nnz, "uniform"))
            F = abi.Factors(ctx, dims, R)
            for k, u in enumerate(_factors(g, dims, R)):
                F.set(k, u.cpu().numpy())
            S = abi.Sampler(ctx, F, abi.EX_SAMPLER_CP_ARLS_LEV, _precision(case), seed=s)
            A = abi.ALS(ctx, T, F, S, precision=_precision(case))
            A.init()
            members.append((A, F, dims, R))
        B = abi.Batch([m[0] for m in members], case["J"])
        total = sum(sum(d) * R for _, _, d, R in members)
        return dict(case=case, batch=B, members=members, out=torch.empty(total, dtype=torch.float64, pin_memory=True))
    g, dims, coords, vals = _raw(case, seed)
    if case["kind"] == "step":
        U = _factors_under_way(g, dims, case["R"], coords)
    else:
        U = _factors(g, dims, case["R"])
    if case["kind"] == "adjoint":
        T = _tensor(ctx, dims, coords, vals)
        T.build_lookups()
        samples, weights, G = _adjoint_inputs(g, case, dims, coords)
        U = [u.requires_grad_(k != case["mode"]) for k, u in enumerate(U)]
        return dict(case=case, T=T, U=U, samples=samples, weights=weights, G=G)
    T = _tensor(ctx, dims, coords, vals)
    del coords, vals
    F = abi.Factors(ctx, dims, case["R"])
    U0 = [_host(u) for u in U]
    for k, u in enumerate(U0):
        F.set(k, u.numpy())
    state = dict(case=case, F=F, U0=U0, out=[torch.empty_like(u, pin_memory=True) for u in U0])
    if case["kind"] == "exact":
        A = abi.ALS.exact(ctx, T, F, precision=_precision(case))
    else:
        state["S"] = _sampler(ctx, case, F, seed)
        A = abi.ALS(ctx, T, F, state["S"], precision=_precision(case))
        if case.get("graph"):
            A.use_graph(True)
    A.init()
    state["A"] = A
    return state


def _adjoint_inputs(g, case, dims, coords):
    """Distinct sample tuples (leverage sampling lands on the tensor's fibers:
    those of random nonzeros), their weights, and an output gradient."""
    mode, J = case["mode"], min(case["J"], case["nnz"])
    pick = coords[torch.randint(coords.shape[0], (J,), generator=g, device="cuda")].clone()
    pick[:, mode] = 0
    key = _keys(pick, dims, mode)
    order = torch.unique(key, return_inverse=True)[1]
    first = torch.full((int(order.max()) + 1,), J, dtype=torch.int64, device="cuda")
    first.scatter_reduce_(0, order, torch.arange(J, device="cuda"), "amin")
    samples = pick[first.sort()[0]].to(torch.int32).contiguous()
    weights = 0.5 + torch.rand(samples.shape[0], generator=g, device="cuda", dtype=torch.float64)
    G = torch.randn((dims[mode], case["R"]), generator=g, device="cuda", dtype=torch.float64)
    return samples, weights, G


def _keys(coords, dims, mode):
    key = torch.zeros(coords.shape[0], dtype=torch.int64, device=coords.device)
    for k, d in enumerate(dims):
        if k != mode:
            key = key * d + coords[:, k].long()
    return key


# ---------------------------------------------------------------- one pass
def _read(F, k, buf):
    """Factor k into the program's own host buffer."""
    abi.check(abi.lib().ex_factors_get(F.h, k, ctypes.cast(buf.data_ptr(), ctypes.POINTER(ctypes.c_double))))
    return buf


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "batch":
        state["batch"].run(case["sweeps"])
        at = 0
        for _, F, dims, R in state["members"]:
            for k, d in enumerate(dims):
                _read(F, k, state["out"][at:at + d * R])
                at += d * R
        return {"factors": state["out"], "sigma": [F.sigma() for _, F, _, _ in state["members"]][0]}
    if kind == "adjoint":
        U, mode = state["U"], case["mode"]
        Y = autograd.SampledMTTKRP.apply(state["T"], mode, state["samples"], state["weights"], *U)
        grads = torch.autograd.grad(Y, [u for k, u in enumerate(U) if k != mode], state["G"])
        return {"Y": Y, "grads": list(grads)}
    F, A = state["F"], state["A"]
    if kind == "step":
        # factors are FP32 on this path: the program keeps them as such
        A.step(case["mode"], case["J"], 1)
        u = _read(F, case["mode"], state["out"][case["mode"]])
        return {"factor": u.float(), "sigma": F.sigma().astype(np.float32)}
    for k, u in enumerate(state["U0"]):
        F.set(k, u.numpy())
    if kind == "exact":
        A.run(case["sweeps"], 1, epoch=case["sweeps"] + 1)
    else:
        for k in range(F.N):
            state["S"].update(k)
        A.run(case["sweeps"], case["J"], epoch=case["sweeps"])
    out = [_read(F, k, buf) for k, buf in enumerate(state["out"])]
    if case["precision"] == "mixed":
        return {"factors": [u.float() for u in out], "sigma": F.sigma().astype(np.float32)}
    got = {"factors": out, "sigma": F.sigma()}
    if kind == "run":
        fit = json.loads(A.stats_json())["fits"][-1]
        got["residual"] = math.nan if fit is None else 1.0 - fit   # of the exact fit
    return got


# ---------------------------------------------------------------- what a pass cannot do without
def _step_work(dims, nnz, R, J, j, s, sts):
    """One randomized mode step: sample state read (a tree path or a search
    per draw), samples and weights, the sampled factor rows, the nonzeros of
    the sampled fibers (at least one coordinate tuple and value per sample
    that hits), the target factor written, the sampler state over it built."""
    N = len(dims)
    hits = min(nnz, J * max(1.0, nnz / (math.prod(dims) / dims[j])))
    bytes_ = J * (4 * N + 8) * 2 + J * (N - 1) * R * s + hits * (4 * N + s) + 2 * dims[j] * R * s
    flops = 2 * J * R * R + 2 * hits * R + 4 * dims[j] * R * R
    if sts:
        tri = R * (R + 1) // 2
        for k, d in enumerate(dims):
            if k != j:
                levels = max(1, math.ceil(math.log2(max(2, d / R)))) + max(1, math.ceil(math.log2(R)))
                bytes_ += min(J, d // R + 1) * (2 * tri + R * R) * s
                flops += J * (levels * 2 * tri + 2 * R * R)
        bytes_ += 2 * (dims[j] // R + 1) * tri * s
        flops += dims[j] * R * R
    else:
        bytes_ += dims[j] * 16 + J * (N - 1) * 16
        flops += 2 * dims[j] * R * R
    return bytes_, flops


def work(case):
    s = 4 if case["precision"] == "mixed" else 8
    if case["kind"] == "batch":
        b = f = 0.0
        for dims, nnz, R, _ in _batch_tensors(case, 0):
            for j in range(3):
                x, y = _step_work(dims, nnz, R, case["J"], j, s, False)
                b, f = b + x * case["sweeps"], f + y * case["sweeps"]
        return {"bytes": b, "flops": f}
    dims, nnz, R = _dims(case), case["nnz"], case["R"]
    N = len(dims)
    if case["kind"] == "step":
        b, f = _step_work(dims, nnz, R, case["J"], case["mode"], s, case["sampler"] == "sts")
        return {"bytes": b, "flops": f}
    if case["kind"] == "adjoint":
        J, j = case["J"], case["mode"]
        hits = J * max(1.0, nnz / (math.prod(dims) / dims[j]))
        rows = sum(d for k, d in enumerate(dims) if k != j)
        return {"bytes": 2 * J * (4 * N + 8 + (N - 1) * R * 8) + 2 * hits * (4 * N + 8 + 8 * R) + dims[j] * R * 8
                + rows * R * 8, "flops": 2 * (2 * hits * R + 2 * J * N * R)}
    ends = 2 * sum(dims) * R * 8   # the factors in and out
    if case["kind"] == "exact":
        b = f = 0.0
        for j in range(N):
            b += nnz * (4 * N + s) + 2 * dims[j] * R * s + sum(d for k, d in enumerate(dims) if k != j) * R * s
            f += nnz * R * N + 4 * dims[j] * R * R
        return {"bytes": b * case["sweeps"] + ends, "flops": f * case["sweeps"]}
    b = f = 0.0
    for j in range(N):
        x, y = _step_work(dims, nnz, R, case["J"], j, s, case["sampler"] == "sts")
        b, f = b + x * case["sweeps"], f + y * case["sweeps"]
    fit = nnz * (4 * N + 8) + sum(dims) * R * 8
    return {"bytes": b + ends + fit, "flops": f + nnz * R * (N + 1)}


# ---------------------------------------------------------------- the same in 64 bits
def _exact_adjoint(case, seed):
    g, dims, coords, vals = _raw(case, seed)
    U = _factors(g, dims, case["R"])
    samples, weights, G = _adjoint_inputs(g, case, dims, coords)
    mode, R = case["mode"], case["R"]
    others = [k for k in range(len(dims)) if k != mode]
    rows = [U[k][samples[:, k].long()] for k in others]
    D = weights[:, None].expand(-1, R)
    for u in rows:
        D = D * u
    key, order = _keys(samples, dims, mode).sort()
    nz = _keys(coords, dims, mode)
    at = torch.searchsorted(key, nz).clamp_(max=key.numel() - 1)
    hit = key[at] == nz
    c, i, x = order[at[hit]], coords[hit, mode], vals[hit]
    Y = torch.zeros((dims[mode], R), dtype=torch.float64, device="cuda").index_add_(0, i, x[:, None] * D[c])
    dD = torch.zeros_like(D.contiguous()).index_add_(0, c, x[:, None] * G[i])
    grads = []
    for q, k in enumerate(others):
        d = dD * weights[:, None]
        for q2, u in enumerate(rows):
            if q2 != q:
                d = d * u
        grads.append(torch.zeros_like(U[k]).index_add_(0, samples[:, k].long(), d))
    return {"Y": Y, "grads": grads}


def _exact_als(case, seed):
    g, dims, coords, vals = _raw(case, seed)
    U = _factors(g, dims, case["R"])
    R = case["R"]
    sigma = None
    for _ in range(case["sweeps"]):
        for j in range(len(dims)):
            H = torch.ones((R, R), dtype=torch.float64, device="cuda")
            Y = torch.zeros((dims[j], R), dtype=torch.float64, device="cuda")
            for k in range(len(dims)):
                if k != j:
                    H = H * (U[k].T @ U[k])
            for a in range(0, coords.shape[0], 1 << 21):
                c = coords[a:a + (1 << 21)]
                p = vals[a:a + (1 << 21), None].expand(-1, R)
                for k in range(len(dims)):
                    if k != j:
                        p = p * U[k][c[:, k]]
                Y.index_add_(0, c[:, j], p)
            lam, V = torch.linalg.eigh(H.cpu())
            inv = torch.where(lam > 1e-11, 1.0 / lam, torch.zeros_like(lam))
            V = V.cuda()
            u = Y @ ((V * inv.cuda()) @ V.T)
            sigma = u.norm(dim=0)
            U[j] = u / sigma
    return {"factors": U, "sigma": sigma}


def exact(case, seed):
    if case["kind"] == "adjoint":
        return _exact_adjoint(case, seed)
    if case["kind"] == "exact":
        return _exact_als(case, seed)
    return None   # the draws are the library's own generator's
