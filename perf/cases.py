"""Timed cases of the CP decomposition library: what its users run, through the public Python entry points.

listed()            the named cases
draw(rng)           one more case of the same ranges
prepare(case, seed) the inputs of a case on the GPU, and the handles a program keeps
run(state)          one pass through the entry points
work(case)          the bytes and operations that a pass cannot do without
exact(case, seed)   the same outputs in 64 bits, in plain torch

A case is a dict: "op" names the entry point, "shape" the tensor ("256x256x256"), "rank" the CP rank, and further
keys the options of that entry point.  Dense tensors are CP models with noise (unit-norm factor columns, weights
U(0.5, 2)); sparse ones have Zipf(1.2) indices over a permutation of each mode and values U(0, 1), like the workloads
of tenrso_amd.synth, drawn on the GPU here.
"""
import math

import numpy as np
import torch

from tenrso_amd import ad, decomp, kernels
from tenrso_amd.sparse import SparseTensor

DEV = "cuda"


def listed():
    return [
        # The smallest tensor of the benchmark: a call is launches and host work.
        {"name": "mttkrp_64_r8", "op": "mttkrp", "shape": "64x64x64", "rank": 8, "dtype": "f32"},
        # The headline tensor: every mode's MTTKRP, the drop-in call that dominates a CP decomposition.
        {"name": "mttkrp_256_r64", "op": "mttkrp", "shape": "256x256x256", "rank": 64, "dtype": "f32"},
        # A ragged size: rows that no vector or tile divides.
        {"name": "mttkrp_250_r64", "op": "mttkrp", "shape": "250x250x250", "rank": 64, "dtype": "f32"},
        # A 4-way tensor of 340 MB: the MTTKRP that streams memory.
        {"name": "mttkrp_96x4_r32", "op": "mttkrp", "shape": "96x96x96x96", "rank": 32, "dtype": "f32"},
        # The bf16 tensor option, on the largest 3-way tensor of the benchmark.
        {"name": "mttkrp_bf16_512_r64", "op": "mttkrp", "shape": "512x512x128", "rank": 64, "dtype": "bf16"},
        # Backward of the MTTKRP: the gradients of the tensor (a reconstruction) and of the other factors.
        {"name": "vjp_256_r64", "op": "vjp", "shape": "256x256x256", "rank": 64, "mode": 1},
        # The CP loss and its gradients, a step of a user's own optimiser.
        {"name": "loss_grad_96x4_r32", "op": "loss_grad", "shape": "96x96x96x96", "rank": 32},
        # The whole decomposition at the headline size in both precisions.
        {"name": "als_256_r64", "op": "als", "shape": "256x256x256", "rank": 64, "iters": 10, "precision": "fp32"},
        {"name": "als_bf16_256_r64", "op": "als", "shape": "256x256x256", "rank": 64, "iters": 10, "precision": "bf16"},
        # ... and at the largest rank that it takes, where the normal equations outweigh the MTTKRP.
        {"name": "als_256_r128", "op": "als", "shape": "256x256x256", "rank": 128, "iters": 5, "precision": "fp32"},
        # The sparse MTTKRP of every mode, 20 million nonzeros.
        {"name": "sparse_20m_r32", "op": "sparse", "shape": "10000x8000x6000", "nnz": 20000000, "rank": 32},
        # The SVD-based initial factors that a decomposition may start from.
        {"name": "svd_init_256_r64", "op": "init", "shape": "256x256x256", "rank": 64},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _sizes(rng, nd, lo, hi, most):
    """Mode sizes over their logarithm, odd ones and multiples of 32 alike, at most `most` elements."""
    while True:
        s = [_log(rng, lo, hi) for _ in range(nd)]
        if rng.random() < 0.4:
            s = [max(32, (n + 16) // 32 * 32) for n in s]
        if math.prod(s) <= most:
            return s


def draw(rng):
    op = rng.choice(["mttkrp", "mttkrp", "mttkrp", "vjp", "loss_grad", "als", "als", "sparse", "init"])
    if op == "sparse":
        nd = rng.choice([3, 3, 4])
        s = [_log(rng, 200, 10000) if nd == 3 else _log(rng, 60, 1000) for _ in range(nd)]
        nnz = min(_log(rng, 20000, 20000000), math.prod(s) // 50)
        return {"op": op, "shape": "x".join(map(str, s)), "nnz": nnz, "rank": rng.choice([4, 8, 10, 16, 25, 32, 48, 64])}
    nd = rng.choice([3, 3, 4])
    lo, hi = (24, 512) if nd == 3 else (12, 96)
    c = {"op": op}
    if op == "mttkrp":
        s = _sizes(rng, nd, lo, hi, 1 << 25)
        c |= {"rank": _log(rng, 4, 96), "dtype": rng.choice(["f32", "f32", "bf16"])}
    elif op == "vjp":
        s = _sizes(rng, nd, lo, hi, 1 << 24)
        c |= {"rank": _log(rng, 4, 96), "mode": rng.randrange(nd)}
    elif op == "loss_grad":
        s = _sizes(rng, nd, lo, hi, 1 << 25)
        c |= {"rank": _log(rng, 4, 64)}
    elif op == "als":
        s = _sizes(rng, nd, lo, 256 if nd == 3 else 64, 1 << 24)
        c |= {"rank": min(_log(rng, 4, 128), min(s) // 2), "iters": rng.randint(3, 8), "precision": rng.choice(["fp32", "bf16"])}
    else:
        s = _sizes(rng, nd, lo, 256 if nd == 3 else 64, 1 << 24)
        c |= {"rank": min(_log(rng, 4, 64), min(s))}
    return {"op": c.pop("op"), "shape": "x".join(map(str, s)), **c}


def _shape(case):
    return tuple(int(n) for n in case["shape"].split("x"))


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _kr(factors):
    """Khatri-Rao rows of the factors, the last one fastest."""
    k = factors[0]
    for f in factors[1:]:
        k = (k[:, None, :] * f[None, :, :]).reshape(-1, f.shape[1])
    return k


def _dense(case, seed):
    """The tensor and a set of factors N(0, 1), such as a decomposition starts from."""
    shape, rank = _shape(case), case["rank"]
    g = _gen(seed)
    model = [torch.randn(n, rank, generator=g, device=DEV) for n in shape]
    model = [f / f.norm(dim=0, keepdim=True) for f in model]
    w = 0.5 + 1.5 * torch.rand(rank, generator=g, device=DEV)
    h = len(shape) // 2
    X = ((_kr(model[:h]) * w) @ _kr(model[h:]).t().contiguous()).reshape(shape)
    X += 1e-3 * torch.randn(shape, generator=g, device=DEV)
    return X, [torch.randn(n, rank, generator=g, device=DEV) for n in shape], g


def _coo(case, seed):
    """Unique coordinates in order (int32, one row a mode), values, and the factors."""
    shape, nnz, g = _shape(case), case["nnz"], _gen(seed)
    perms = [torch.randperm(n, generator=g, device=DEV) for n in shape]
    cdfs = [torch.cumsum(torch.arange(1, n + 1, dtype=torch.float64, device=DEV) ** -1.2, 0) for n in shape]
    keys = torch.empty(0, dtype=torch.int64, device=DEV)
    while keys.numel() < nnz:
        lin = torch.zeros(2 * nnz, dtype=torch.int64, device=DEV)
        for n, perm, cdf in zip(shape, perms, cdfs):
            u = torch.rand(2 * nnz, generator=g, device=DEV, dtype=torch.float64) * cdf[-1]
            lin = lin * n + perm[torch.searchsorted(cdf, u).clamp_(max=n - 1)]
        keys = torch.unique(torch.cat([keys, lin]))
    keep = torch.randperm(keys.numel(), generator=g, device=DEV)[:nnz]
    keys = keys[keep.sort().values]
    idx = torch.empty(len(shape), nnz, dtype=torch.int32, device=DEV)
    for k in range(len(shape) - 1, -1, -1):
        idx[k] = (keys % shape[k]).to(torch.int32)
        keys = keys // shape[k]
    vals = torch.rand(nnz, generator=g, device=DEV)
    return idx, vals, [torch.randn(n, case["rank"], generator=g, device=DEV) for n in shape]


def prepare(case, seed):
    op = case["op"]
    if op == "sparse":
        idx, vals, F = _coo(case, seed)
        return {"case": case, "sp": SparseTensor(idx.cpu().numpy(), vals.cpu().numpy(), _shape(case)), "F": F}
    X, F, g = _dense(case, seed)
    state = {"case": case, "X": X, "F": F}
    if op == "mttkrp" and case["dtype"] == "bf16":
        state["X"] = X.to(torch.bfloat16)
    if op == "vjp":
        state["rule"] = ad.MttkrpVjp(X, F, case["mode"])
        state["grad"] = torch.randn(F[case["mode"]].shape, generator=g, device=DEV)
    return state


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "sparse":
        return [state["sp"].mttkrp(state["F"], m) for m in range(len(state["F"]))]
    X, F = state["X"], state["F"]
    if op == "mttkrp":
        if case["dtype"] == "bf16":
            return [kernels.mttkrp_bf16(X, F, m) for m in range(X.dim())]
        return kernels.mttkrp_all_modes(X, F)
    if op == "vjp":
        return state["rule"].vjp(state["grad"])
    if op == "loss_grad":
        return ad.cp_loss_and_grad(X, F)
    if op == "als":
        cp = decomp.cp_als_with_init(X, F, case["iters"], 0.0, precision=case["precision"])
        return {"factors": cp.factors, "fit": cp.fit, "iters": cp.iters}
    return decomp.initialize_factors(X.shape, case["rank"], decomp.InitStrategy.Svd, seed=0, tensor=X)


def work(case):
    op, shape, r = case["op"], _shape(case), case["rank"]
    nd, total, rows = len(shape), math.prod(shape), sum(shape)
    if op == "sparse":
        # per mode: every nonzero's coordinates and value once, the other factors, the result; one product of nd terms and a sum
        nnz = case["nnz"]
        return {"bytes": nd * (4 * (nd + 1) * nnz + 4 * r * rows), "flops": nd * nnz * r * nd}
    if op == "mttkrp":
        return {"bytes": nd * (total * (2 if case["dtype"] == "bf16" else 4) + 4 * r * rows), "flops": nd * 2 * total * r}
    if op == "vjp":
        # the tensor and its gradient, the factors, the cotangent and the gradients; nd - 1 MTTKRPs and a reconstruction
        return {"bytes": 8 * total + 8 * r * rows, "flops": nd * 2 * total * r}
    if op == "loss_grad":
        # two partial MTTKRPs give all modes' products
        return {"bytes": 4 * total + 8 * r * rows, "flops": 2 * 2 * total * r}
    if op == "als":
        # every mode's MTTKRP of every sweep reads the tensor
        return {"bytes": case["iters"] * nd * 4 * total + 8 * r * rows,
                "flops": case["iters"] * (nd * 2 * total * r + sum(2 * n * r * r for n in shape) * 2 + nd * 2 * r**3)}
    # half of every mode's n x n Gram, and its eigenvectors
    return {"bytes": nd * 4 * total + 4 * r * rows, "flops": sum(total * n + 10 * n**3 for n in shape)}


def _mttkrp64(X, F, mode):
    nd = len(F)
    Xn = X.movedim(mode, 0).reshape(X.shape[mode], -1).contiguous()
    return Xn @ _kr([F[k] for k in range(nd) if k != mode])


def _grams(F, skip=None):
    g = None
    for k, f in enumerate(F):
        if k != skip:
            h = f.t().contiguous() @ f
            g = h if g is None else g * h
    return g


def _als64(case, X, F):
    lead = X.to(torch.bfloat16).double() if case["precision"] == "bf16" else X.double()
    X = X.double()
    nd = X.dim()
    norm = float((X * X).sum())
    fit = 0.0
    for _ in range(case["iters"]):
        for n in range(nd):
            M = _mttkrp64(X if n == nd - 1 else lead, F, n)
            F[n] = torch.linalg.solve(_grams(F, n).cpu(), M.t().cpu()).t().contiguous().to(DEV)
        err = norm + float(_grams(F).sum()) - 2.0 * float((M * F[-1]).sum())
        fit = min(1.0, max(0.0, 1.0 - math.sqrt(max(err, 0.0) / norm)))
    return {"factors": F, "fit": fit, "iters": case["iters"]}


def _init64(case, X):
    out = []
    for k in range(X.dim()):
        Xk = X.double().movedim(k, 0).reshape(X.shape[k], -1).contiguous()
        lam, V = np.linalg.eigh((Xk @ Xk.t().contiguous()).cpu().numpy())
        U = V[:, ::-1][:, :case["rank"]]
        U = U * np.sign(U[np.abs(U).argmax(0), np.arange(U.shape[1])])
        out.append(np.ascontiguousarray(U))
    return out


def exact(case, seed):
    op = case["op"]
    if op == "sparse":
        idx, vals, F = _coo(case, seed)
        F = [f.double() for f in F]
        outs = []
        for m in range(len(F)):
            out = torch.zeros_like(F[m])
            for lo in range(0, vals.numel(), 1 << 21):
                t = vals[lo:lo + (1 << 21), None].double().expand(-1, case["rank"])
                for k in range(len(F)):
                    if k != m:
                        t = t * F[k][idx[k, lo:lo + (1 << 21)].long()]
                out.index_add_(0, idx[m, lo:lo + (1 << 21)].long(), t)
            outs.append(out)
        return outs
    X, F, g = _dense(case, seed)
    F64 = [f.double() for f in F]
    if op == "mttkrp":
        X = (X.to(torch.bfloat16) if case["dtype"] == "bf16" else X).double()
        return [_mttkrp64(X, F64, m) for m in range(X.dim())]
    if op == "vjp":
        F64[case["mode"]] = torch.randn(F[case["mode"]].shape, generator=g, device=DEV).double()
        h = X.dim() // 2
        dX = (_kr(F64[:h]) @ _kr(F64[h:]).t().contiguous()).reshape(X.shape)
        return [dX] + [_mttkrp64(X.double(), F64, m) for m in range(X.dim()) if m != case["mode"]]
    if op == "loss_grad":
        X = X.double()
        h = X.dim() // 2
        res = X.reshape(-1) - (_kr(F64[:h]) @ _kr(F64[h:]).t().contiguous()).reshape(-1)
        loss = 0.5 * float((res * res).sum())
        return loss, [F64[n] @ _grams(F64, n) - _mttkrp64(X, F64, n) for n in range(X.dim())]
    if op == "als":
        return _als64(case, X, F64)
    return _init64(case, X)
