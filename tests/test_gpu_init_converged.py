"""The eigenproblem of the SVD-based initial factors where its convergence is hard: tensors without noise (a null
space of rounding noise only), singular values over four decades, more than 300 rows, and a bulk of close
eigenvalues, against numpy.

Tolerances: an entry is rounded to fp32 (2^-24 at most); the FP64 Gram's rounding, some 2^-50 of its norm, over the
smallest gap of these spectra (2e-9 of the norm at weights to 1e-4) leaves less than 2^-22 in all.  Where the
spectrum has no gaps, orthogonality and the residual K u - l u of the rounded vectors need none: 2^-22 of ||K||.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from tenrso_amd import decomp  # noqa: E402


def left_vectors(X, R):
    got = decomp.initialize_factors(X.shape, R, decomp.InitStrategy.Svd, seed=0, tensor=torch.from_numpy(X).cuda())[0]
    return np.asarray(got, dtype=np.float64)


@pytest.mark.parametrize("n,R,low", [(256, 64, None), (256, 64, 1e-3), (256, 64, 1e-4), (512, 128, 1e-3), (1024, 64, 1e-3),
                                     (64, 20, 1e-4), (130, 40, None)])
def test_exact_low_rank(n, R, low):
    print(f"[case] svd init exact rank {n} rows R={R} low={low}", flush=True)
    rng = np.random.default_rng(0)
    F = [rng.standard_normal((k, R)) for k in (n, 64, 64)]
    F = [f / np.linalg.norm(f, axis=0) for f in F]
    w = rng.uniform(0.5, 2.0, R) if low is None else np.geomspace(1.0, low, R)
    X = ((F[0] * w) @ (F[1][:, None] * F[2][None]).reshape(-1, R).T).astype(np.float32)
    want = np.linalg.svd(X.astype(np.float64), full_matrices=False)[0][:, :R]
    want *= np.sign(want[np.argmax(np.abs(want), axis=0), np.arange(R)])
    got = left_vectors(X.reshape(n, 64, 64), R)
    assert np.abs(got - want).max() <= 2.0 ** -22, float(np.abs(got - want).max())


@pytest.mark.parametrize("n,R", [(300, 64), (1000, 128)])
def test_close_eigenvalues(n, R):
    print(f"[case] svd init close eigenvalues {n} rows R={R}", flush=True)
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n, 40, 40)).astype(np.float32)
    U = left_vectors(X, R)
    K = X.reshape(n, -1).astype(np.float64)
    K = K @ K.T
    lam = np.linalg.eigvalsh(K)[::-1]
    assert np.abs(U.T @ U - np.eye(R)).max() <= 2.0 ** -22
    KU = K @ U
    l = (U * KU).sum(0)
    assert np.linalg.norm(KU - U * l, axis=0).max() <= 2.0 ** -22 * lam[0]
    assert np.abs(l - lam[:R]).max() <= 2.0 ** -22 * lam[0]


@pytest.mark.parametrize("n,R,scale", [(96, 64, 1e-6), (64, 50, 1e-8), (300, 80, 1e-7)])
def test_slices_of_two_scales(n, R, scale):
    """Small slices beside ordinary ones: their vectors, which span the small rows up to `scale`, by residual and
    orthogonality, relative to the small part of K.  Rows are multiplied by a power of two, so that the small part is
    exact; what couples the two parts moves it by the large part's projection only, a factor of order one."""
    print(f"[case] svd init two scales {n} rows R={R} scale {scale}", flush=True)
    rng = np.random.default_rng(n)
    big = 20
    X = rng.standard_normal((n, 64, 64)).astype(np.float32)
    p2 = np.float32(2.0 ** np.round(np.log2(scale)))
    X[big:] *= p2
    U = left_vectors(X, R)[big:, big:] * 1.0  # the small rows of the small vectors
    Y = X.reshape(n, -1).astype(np.float64)
    A, B = Y[:big], Y[big:] / float(p2)
    # the small part with the large rows' span taken out: what the small vectors diagonalise, up to p2^2
    B = B - (B @ A.T) @ np.linalg.solve(A @ A.T, A)
    K = B @ B.T
    KU = K @ U
    l = (U * KU).sum(0)
    lam = np.linalg.eigvalsh(K)[::-1][:R - big]
    assert np.abs(U.T @ U - np.eye(R - big)).max() <= 2.0 ** -22
    assert np.linalg.norm(KU - U * l, axis=0).max() <= 2.0 ** -18 * lam[0]
    assert np.abs(l - lam).max() <= 2.0 ** -22 * lam[0]


def test_leading_vector_of_a_constant_tensor():
    print("[case] svd init constant tensor", flush=True)
    U = left_vectors(np.ones((70, 66, 3), np.float32), 3)
    assert np.abs(U[:, 0] - 70 ** -0.5).max() <= 2.0 ** -24
