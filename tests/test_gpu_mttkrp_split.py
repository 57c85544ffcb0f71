"""The fp32 MTTKRP from exact bf16 triples: the edges of its tiles and load forms, and the values at which a
split into bf16 parts could go wrong (infinities, NaN, values that round to infinity in bf16, and scales near
the ends of the exponent range), against FP64.

Tolerance, per element: the J terms of a row are rounded a few times each (the split's remainder, the
Khatri-Rao factor, the product with PRE) and summed in fp32, every rounding at most 2^-23 of the sum of the
magnitudes: (J + 8) 2^-23 sum |x kr|.  With J <= 64 that is below 2^-16, the size of a lost low part.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from tenrso_amd import kernels  # noqa: E402


def mttkrp64(X, F, mode, mag=False):
    X, F = X.astype(np.float64), [f.astype(np.float64) for f in F]
    if mag:
        X, F = np.abs(X), [np.abs(f) for f in F]
    kr = np.ones((1, F[0].shape[1]))
    for k, f in enumerate(F):
        if k != mode:
            kr = (kr[:, None, :] * f[None, :, :]).reshape(-1, f.shape[1])
    return np.moveaxis(X, mode, 0).reshape(X.shape[mode], -1) @ kr


def run(X, F, offset=0):
    flat = torch.empty(X.size + offset, device="cuda")
    flat[offset:] = torch.from_numpy(np.ascontiguousarray(X)).cuda().reshape(-1)
    Xd = flat[offset:].view(X.shape)
    Fd = [torch.from_numpy(f).cuda() for f in F]
    return [kernels.mttkrp(Xd, Fd, m).cpu().numpy() for m in range(X.ndim)]


def check(X, F, got):
    for m in range(X.ndim):
        J = X.size // X.shape[m]
        lim = (J + 8) * 2.0 ** -23 * mttkrp64(X, F, m, mag=True) + 1e-44
        d = np.abs(got[m] - mttkrp64(X, F, m))
        assert np.all(d <= lim), (m, float((d / lim).max()))


# last modes of one row, odd last modes (pairs of rows with a single last one), windows with a partial last
# block, two windows, tensors of fewer elements than a vector, more row tiles than the GPU holds at once
SHAPES = [((1, 2), 1), ((3, 1), 2), ((2, 2, 1), 3), ((5, 7, 1), 16), ((1, 9, 33), 17), ((31, 4, 3), 4), ((33, 2, 31), 8),
          ((32, 2, 32), 64), ((34, 3, 63), 20), ((65, 2, 129), 33), ((3, 130, 35), 48), ((4, 3, 5, 67), 12),
          ((9000, 2, 20), 8), ((2, 20, 9001), 5), ((3, 9004, 2), 36), ((2, 3, 161), 65), ((33, 5, 40), 100),
          ((35, 4, 33), 127), ((6, 20, 32), 128), ((34, 3, 35), 130)]


@pytest.mark.parametrize("offset", [0, 1, 2])
@pytest.mark.parametrize("shape,R", SHAPES)
def test_forms_vs_fp64(shape, R, offset):
    print(f"[case] split mttkrp {shape} R={R} offset={offset}", flush=True)
    rng = np.random.default_rng(sum(shape) + R)
    X = rng.standard_normal(shape).astype(np.float32)
    F = [rng.standard_normal((n, R)).astype(np.float32) for n in shape]
    check(X, F, run(X, F, offset))


# (scale of X, scales of the factors): products from the smallest to the largest exponents
SCALES = [(1e-30, (1.0, 1.0, 1.0)), (1e-36, (1.0, 1.0, 1.0)), (1e-37, (1e5, 1.0, 1.0)), (1.0, (1e-34, 1e-3, 1e2)),
          (1e-20, (1e-18, 1e10, 1e12)), (1e-20, (1e10, 1e-18, 1e12)), (1e30, (1e3, 1e3, 1e-3)), (1e38, (1.0, 1e-3, 1e-3)),
          (1e-25, (1e15, 1e15, 1e-5))]


@pytest.mark.parametrize("xs,fs", SCALES)
def test_scales_vs_fp64(xs, fs):
    """Every mode whose result and Khatri-Rao rows are normal fp32 numbers keeps the tolerance of scale 1."""
    print(f"[case] split mttkrp scale {xs} {fs}", flush=True)
    rng = np.random.default_rng(3)
    shape, R = (34, 2, 32), 20
    X = (rng.uniform(0.5, 2.0, shape) * xs * rng.choice([-1, 1], shape)).astype(np.float32)
    F = [(rng.uniform(0.5, 2.0, (n, R)) * s).astype(np.float32) for n, s in zip(shape, fs)]
    got = run(X, F)
    for m in range(3):
        J = X.size // shape[m]
        kr = np.prod([s for k, s in enumerate(fs) if k != m])
        if not (1e-36 < kr < 1e36 and 1e-36 < xs * kr < 1e35):
            continue
        lim = (J + 8) * 2.0 ** -23 * mttkrp64(X, F, m, mag=True)
        assert np.all(np.abs(got[m] - mttkrp64(X, F, m)) <= lim), m


def test_rows_of_very_different_scale():
    print("[case] split mttkrp mixed row scales", flush=True)
    rng = np.random.default_rng(5)
    shape, R = (40, 2, 31), 9
    X = rng.standard_normal(shape).astype(np.float32)
    X[3] *= np.float32(1e-35)
    X[7] = 0.0
    X[:, :, 5] *= np.float32(1e-36)
    F = [rng.uniform(0.5, 1.5, (n, R)).astype(np.float32) for n in shape]
    F[2][:, 4] *= np.float32(1e-33)
    F[1][:, 6] = 0.0
    got = run(X, F)
    check(X, F, got)
    assert np.all(got[0][7] == 0.0) and np.all(got[0][:, 6] == 0.0)


@pytest.mark.parametrize("shape", [(34, 2, 32), (35, 3, 33), (9000, 2, 20)])
def test_infinities_and_nan(shape):
    """As fp32 arithmetic gives them: an infinity in X with factors that are not zero makes its rows infinite
    with the sign of the product, with a zero factor or two opposite infinities NaN; the largest finite values
    (which round to infinity in bf16) stay finite."""
    print(f"[case] split mttkrp infinities {shape}", flush=True)
    rng = np.random.default_rng(7)
    R = 6
    X = rng.uniform(0.5, 1.0, shape).astype(np.float32)
    F = [rng.uniform(0.5, 1.0, (n, R)).astype(np.float32) for n in shape]
    F[1][0] *= -1
    X[4, 0, 3] = np.inf
    X[6, 1, 2] = -np.inf
    X[8, 0, 1], X[8, 1, 1] = np.inf, np.inf
    X[9, 0, 0] = np.nan
    X[10, 0, :] = 0.0
    X[10, 0, 5] = np.float32(3.4028235e38)
    F[2][5] *= np.float32(0.25)
    got = run(X, F)
    with np.errstate(all="ignore"):
        for m in range(3):
            ref = mttkrp64(X, F, m)
            assert np.array_equal(np.isnan(got[m]), np.isnan(ref)), m
            big = np.isinf(ref)
            assert np.array_equal(got[m][big], ref[big].astype(np.float32)), m
            fin = np.isfinite(ref)
            mag = mttkrp64(np.where(np.isfinite(X), X, 0), F, m, mag=True)
            J = X.size // shape[m]
            ok = np.abs(got[m] - ref) <= (J + 8) * 2.0 ** -23 * mag
            assert np.all(ok[fin & (mag < 3e38)]), m
