"""The wide-rank normal equations (ranks 65 to 128) on their own: one ALS update per mode against the FP64
solution of the same normal equations, at ranks that end inside a pivot block, a strip of 16 and the last strip.

Tolerance: the row solve and the inverse are FP64; the MTTKRP's fp32 error (a relative 2^-21 of each row at
these sizes) and the fp32 factors it is computed from are amplified by at most the condition number of Gamma.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from tenrso_amd import decomp  # noqa: E402


@pytest.mark.parametrize("R", [65, 67, 80, 81, 96, 97, 112, 113, 116, 120, 124, 127, 128])
def test_one_update_per_mode_vs_fp64(R):
    print(f"[case] wide inverse R={R}", flush=True)
    rng = np.random.default_rng(R)
    shape = (R + 40, R + 60, R + 50)
    F = [rng.standard_normal((n, R)) for n in shape]
    X = np.einsum("ir,jr,kr->ijk", *F, optimize=True) + rng.standard_normal(shape)
    X = X.astype(np.float32)
    init = [rng.standard_normal((n, R)).astype(np.float32) for n in shape]
    cp = decomp.cp_als_with_init(torch.from_numpy(X).cuda(), [torch.from_numpy(f).cuda() for f in init], 1, 0.0)
    A = [f.astype(np.float64) for f in init]
    worst = 1.0
    for n in range(3):
        a, b = [k for k in range(3) if k != n]
        G = (A[a].T @ A[a]) * (A[b].T @ A[b])
        worst = max(worst, np.linalg.cond(G))
        M = np.einsum("ijk,jr,kr->ir", np.moveaxis(X.astype(np.float64), n, 0), A[a], A[b], optimize=True)
        want = np.linalg.solve(G, M.T).T
        got = cp.factors[n].cpu().numpy().astype(np.float64)
        err = np.linalg.norm(got - want) / np.linalg.norm(want)
        assert err <= 2.0 ** -21 * worst, (n, err, worst)
        A[n] = got
    assert cp.solve_path_max == 0
