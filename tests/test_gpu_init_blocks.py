"""SVD initial factors at the edges of the eigenvalue kernel's blocks (32 rows a block, 64 a pair; two blocks are
solved at once, more in rounds) against numpy.

X = U diag(2^-k) V^T exactly representable enough that its leading eight singular values are a factor of two
apart: an eigenvector of X X^T is then off by at most some n 2^-53 / 2^-16 in 64-bit arithmetic (1e-9 at 300
rows), and by 2^-24 from its rounding to fp32.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from tenrso_amd import decomp  # noqa: E402


@pytest.mark.parametrize("n", [2, 31, 32, 33, 63, 64, 65, 96, 127, 128, 129, 200, 257, 300])
def test_left_vectors(n):
    print(f"[case] svd init {n} rows", flush=True)
    rng = np.random.default_rng(n)
    R = min(8, n)
    U = np.linalg.qr(rng.standard_normal((n, R)))[0]
    V = np.linalg.qr(rng.standard_normal((96, R)))[0]
    X = ((U * 2.0 ** -np.arange(R)) @ V.T).astype(np.float32).reshape(n, 24, 4)
    got = decomp.initialize_factors(X.shape, R, decomp.InitStrategy.Svd, seed=0, tensor=torch.from_numpy(X).cuda())[0]
    want = np.linalg.svd(X.reshape(n, -1).astype(np.float64))[0][:, :R]
    want *= np.sign(want[np.argmax(np.abs(want), axis=0), np.arange(R)])
    g = np.asarray(got, dtype=np.float64)
    g = g / np.linalg.norm(g, axis=0)
    assert np.all(np.abs(g - want) <= 2.0 ** -22), float(np.abs(g - want).max())


def test_zero_and_constant_tensors():
    """No rotation at all, and one eigenvalue: finite factors."""
    for X in (torch.zeros((70, 5, 3), device="cuda"), torch.ones((70, 66, 3), device="cuda")):
        for f in decomp.initialize_factors(tuple(X.shape), 3, decomp.InitStrategy.Svd, seed=0, tensor=X):
            assert np.all(np.isfinite(np.asarray(f)))
