"""The wide-rank normal equations (ranks 65 to 128) with groups of four nearly collinear columns, where a pivot
block is close to singular: one ALS update of the first mode against the normal equations themselves.

A solution is checked by its residual, which does not grow with the condition: A Gamma = M holds up to the rounding
of A to fp32 (2^-24 of A, times Gamma) and the MTTKRP's fp32 error (2^-21 of M at these sizes); the factor of two of
the tolerance is for the solution itself.  Scalar elimination in FP64 leaves 1e-10 at a condition of 1e7, and takes
Gamma for positive definite up to 1e9.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from tenrso_amd import decomp  # noqa: E402


@pytest.mark.parametrize("d", [1e-2, 1e-3, 1e-4])
@pytest.mark.parametrize("R", [65, 96, 128])
def test_nearly_collinear_groups(R, d):
    print(f"[case] wide pivots R={R} d={d}", flush=True)
    rng = np.random.default_rng(R)
    shape = (R + 12, R + 60, R + 50)
    init = [rng.standard_normal((n, R)) for n in shape]
    for f in init[1:]:
        for g in range(0, R - 4, 16):
            f[:, g + 1:g + 4] = f[:, g:g + 1] + d * rng.standard_normal((f.shape[0], 3))
    init = [f.astype(np.float32) for f in init]
    A = [f.astype(np.float64) for f in init]
    X = np.einsum("ir,jr,kr->ijk", *A, optimize=True).astype(np.float32)
    cp = decomp.cp_als_with_init(torch.from_numpy(X).cuda(), [torch.from_numpy(f).cuda() for f in init], 1, 0.0)
    G = (A[1].T @ A[1]) * (A[2].T @ A[2])
    M = np.einsum("ijk,jr,kr->ir", X.astype(np.float64), A[1], A[2], optimize=True)
    got = cp.factors[0].cpu().numpy().astype(np.float64)
    lim = 2 * (2.0 ** -24 * np.linalg.norm(got) * np.linalg.norm(G) + 2.0 ** -21 * np.linalg.norm(M))
    assert np.linalg.norm(got @ G - M) <= lim, (np.linalg.norm(got @ G - M) / lim, np.linalg.cond(G))
    assert cp.solve_path_max == 0, np.linalg.cond(G)
