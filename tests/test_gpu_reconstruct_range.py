"""CP reconstruction where the product of some of the factors leaves the exponent range and the whole product,
taken from left to right, does not: against the FP64 oracle.

Tolerance: as in the tests of the tiles, (nd + 1 + R) 2^-24 times the sum of the magnitudes: every partial product
from left to right is a normal fp32 number here.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import oracle  # noqa: E402
from tenrso_amd.kernels import cp_reconstruct  # noqa: E402

SCALES = [((1e30, 1e-25, 1e-25), 1.0), ((1e30, 1e-20, 1e-20), 1.0), ((1e-30, 1e22, 1e22), 1.0), ((1e30, 1e-20, 1e-15), 1e20),
          ((1e30, 1e-10, 1e-25, 1e-25), 1e10), ((1e-30, 1e10, 1e20, 1e20), 1e-3), ((1.0, 1e-25, 1e-10), 1.0)]


@pytest.mark.parametrize("R", [5, 20, 68])
@pytest.mark.parametrize("scales,w", SCALES)
def test_partial_products_out_of_range(scales, w, R):
    print(f"[case] reconstruct scales {scales} w={w} R={R}", flush=True)
    rng = np.random.default_rng(R)
    shape = (70, 33, 66) if len(scales) == 3 else (20, 9, 11, 14)
    F = [(rng.uniform(0.5, 2.0, (n, R)) * s).astype(np.float32) for n, s in zip(shape, scales)]
    F[0][3, 1], F[-1][4, 2], F[1][2, :] = 0.0, 0.0, 0.0
    wv = (rng.uniform(0.5, 2.0, R) * w).astype(np.float32)
    F64, w64 = [f.astype(np.float64) for f in F], wv.astype(np.float64)
    got = cp_reconstruct([torch.from_numpy(f).cuda() for f in F], torch.from_numpy(wv).cuda()).cpu().numpy()
    lim = (len(F) + 1 + R) * 2.0 ** -24 * oracle.cp_reconstruct(F64, w64)
    assert np.all(np.abs(got - oracle.cp_reconstruct(F64, w64)) <= lim)
