"""Sparse MTTKRP at the edges of its runs of nonzeros and of the levels that add their carries, against FP64.

Tolerance per element: the n nonzeros of a row are each rounded a few times and added in fp32 within a run, in
FP64 between runs but for one rounding a level, every rounding at most 2^-23 of the sum of the magnitudes:
(n + 16) 2^-23 sum |v f g|, with n at most a run (1024).
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from tenrso_amd.sparse import SparseTensor  # noqa: E402


def reference(idx, vals, F, mode, mag=False):
    f = [x.double().abs() if mag else x.double() for x in F]
    t = (vals.double().abs() if mag else vals.double())[:, None].expand(-1, F[0].shape[1]).clone()
    for k in range(len(F)):
        if k != mode:
            t *= f[k][idx[:, k]]
    out = torch.zeros((F[mode].shape[0], F[0].shape[1]), dtype=torch.float64, device=t.device)
    return out.index_add_(0, idx[:, mode], t)


# one row for all (a carry in every run), a row a nonzero, and rows of a few
@pytest.mark.parametrize("shape", [(1, 300, 400), (70000, 30, 40), (500, 40, 30, 20)])
@pytest.mark.parametrize("nnz,R", [(1, 3), (31, 4), (33, 25), (64, 64), (1023, 10), (1025, 32), (33000, 25), (40000, 16),
                                   (110000, 8), (300000, 32), (300000, 10)])
def test_runs_vs_fp64(shape, nnz, R):
    print(f"[case] sparse runs {shape} nnz={nnz} R={R}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(nnz + R)
    total = int(np.prod(shape))
    flat = torch.randperm(total, generator=g, device="cuda")[:min(nnz, total // 2)]
    cols = []
    for n in reversed(shape):
        cols.append(flat % n)
        flat = flat // n
    idx = torch.stack(cols[::-1], 1)
    vals = torch.randn(idx.shape[0], generator=g, device="cuda")
    F = [torch.randn((n, R), generator=g, device="cuda") for n in shape]
    sp = SparseTensor(idx.t().cpu().numpy(), vals.cpu().numpy(), shape)
    for m in range(len(shape)):
        n = min(1024, int(torch.bincount(idx[:, m]).max()))
        lim = (n + 16) * 2.0 ** -23 * reference(idx, vals, F, m, mag=True) + 1e-30
        assert bool(((sp.mttkrp(F, m).double() - reference(idx, vals, F, m)).abs() <= lim).all()), m
