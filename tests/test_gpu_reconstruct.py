"""CP reconstruction on the matrix cores against the FP64 oracle: the edges of its 64- and 128-wide tiles,
the rank chunks of 16, 32 and 64, every split of the modes, unaligned factors and outputs, and values at
which a zero pad may not turn into NaN.

Tolerance: each element is a sum of R products of at most nd + 1 fp32 roundings, R more roundings of the
sum: (nd + 1 + R) 2^-24 times the sum of the magnitudes.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import oracle  # noqa: E402
from tenrso_amd.kernels import cp_reconstruct  # noqa: E402

SHAPES = [((1,), 1), ((5,), 3), ((300,), 64), ((1, 1, 1), 2), ((63, 65), 16), ((64, 64, 64), 8), ((65, 3, 64), 17),
          ((128, 127, 130), 32), ((129, 128, 128), 33), ((7, 5, 3, 2, 6), 5), ((40, 1, 33, 20), 65), ((2, 2, 4001), 4),
          ((4001, 2, 2), 70), ((1500, 1300), 130), ((3, 2, 2, 2, 2, 2, 2, 3), 6)]


def bound(F, w):
    mags = oracle.cp_reconstruct([np.abs(f) for f in F], None if w is None else np.abs(w))
    return (len(F) + 1 + F[0].shape[1]) * 2.0 ** -24 * mags + 1e-37


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("shape,R", SHAPES)
def test_reconstruct_tiles_vs_oracle(shape, R, weighted):
    print(f"[case] reconstruct {shape} R={R} weighted={weighted}", flush=True)
    rng = np.random.default_rng(sum(shape) + R)
    F = [rng.standard_normal((n, R)).astype(np.float32) for n in shape]
    w = rng.uniform(0.5, 2.0, R).astype(np.float32) if weighted else None
    ref = oracle.cp_reconstruct([f.astype(np.float64) for f in F], None if w is None else w.astype(np.float64))
    wd = None if w is None else torch.from_numpy(w).cuda()
    got = cp_reconstruct([torch.from_numpy(f).cuda() for f in F], wd).cpu().numpy()
    lim = bound([f.astype(np.float64) for f in F], None if w is None else w.astype(np.float64))
    assert got.shape == tuple(shape) and np.all(np.abs(got - ref) <= lim)
    # factors that are only 4-byte aligned (views at an odd offset)
    odd = []
    for f in F:
        t = torch.empty(f.size + 1, device="cuda")
        t[1:] = torch.from_numpy(f).cuda().reshape(-1)
        odd.append(t[1:].view(f.shape))
    got = cp_reconstruct(odd, wd).cpu().numpy()
    assert np.all(np.abs(got - ref) <= lim)


def test_reconstruct_infinities_and_nan_stay_in_their_elements():
    """An infinite or NaN factor row reaches its own elements only (the zero ranks past R meet no pad of it)."""
    print("[case] reconstruct infinities", flush=True)
    rng = np.random.default_rng(1)
    shape, R = (70, 9, 66), 10
    F = [rng.uniform(0.5, 1.5, (n, R)).astype(np.float32) for n in shape]
    F[0][3, 2], F[2][65, 9] = np.inf, np.nan
    got = cp_reconstruct([torch.from_numpy(f).cuda() for f in F]).cpu().numpy()
    want_inf = np.zeros(shape, bool)
    want_inf[3] = True
    want_nan = np.zeros(shape, bool)
    want_nan[:, :, 65] = True
    assert np.array_equal(np.isnan(got), want_nan)
    assert np.array_equal(np.isposinf(got), want_inf & ~want_nan)
