"""The BF16 MTTKRP in each of its load forms (rows of j; four rows of one j; any alignment; partly filled
blocks; the end of X), and values at which bf16 parts of the factors could go wrong, against FP64.

Tolerance: that of the fp32 kernel's tests, since a bf16 element is exact and so are the factors' triples:
(J + 8) 2^-23 sum |x kr| per element.  Calls whose rows are 16-byte aligned vectors take the factor of the
fastest mode as a bf16 pair, off by at most 2^-17 of it.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from test_gpu_mttkrp_split import mttkrp64  # noqa: E402

from tenrso_amd import kernels  # noqa: E402


def bf16(X):
    return torch.from_numpy(np.ascontiguousarray(X)).to(torch.bfloat16)


def run(Xb, F, offset=0):
    flat = torch.empty(Xb.numel() + offset, device="cuda", dtype=torch.bfloat16)
    flat[offset:] = Xb.cuda().reshape(-1)
    Xd = flat[offset:].view(Xb.shape)
    Fd = [torch.from_numpy(f).cuda() for f in F]
    return [kernels.mttkrp_bf16(Xd, Fd, m).cpu().numpy() for m in range(Xb.ndim)]


def as_pair(shape, mode, offset):
    nd = len(shape)
    fast = shape[nd - 2] if mode == nd - 1 else shape[-1]
    return offset % 8 == 0 and fast % 8 == 0 and (mode < nd - 1 or shape[mode] == 1)


def check(X, F, got, offset=0):
    for m in range(X.ndim):
        J = X.size // X.shape[m]
        u = (J + 8) * 2.0 ** -23 + (2.0 ** -17 if as_pair(X.shape, m, offset) else 0.0)
        d = np.abs(got[m] - mttkrp64(X, F, m))
        assert np.all(d <= u * mttkrp64(X, F, m, mag=True) + 1e-44), m


SHAPES = [((1, 2), 1), ((3, 1), 2), ((2, 2, 1), 3), ((5, 7, 1), 16), ((1, 9, 33), 17), ((31, 4, 3), 4), ((33, 2, 31), 8),
          ((32, 2, 64), 64), ((34, 3, 63), 20), ((65, 2, 129), 33), ((3, 130, 35), 48), ((4, 3, 5, 67), 12),
          ((9000, 2, 20), 8), ((2, 20, 9001), 5), ((3, 9004, 2), 36), ((2, 3, 161), 65), ((33, 64, 65), 100),
          ((3, 32, 2), 6), ((2, 31, 3), 7), ((2, 40, 5), 9), ((2, 128, 4), 32), ((3, 96, 66), 64), ((6, 20, 32), 128)]


@pytest.mark.parametrize("offset", [0, 1, 2, 4])
@pytest.mark.parametrize("shape,R", SHAPES)
def test_forms_vs_fp64(shape, R, offset):
    print(f"[case] bf16 forms {shape} R={R} offset={offset}", flush=True)
    rng = np.random.default_rng(sum(shape) + R)
    Xb = bf16(rng.standard_normal(shape).astype(np.float32))
    F = [rng.standard_normal((n, R)).astype(np.float32) for n in shape]
    check(Xb.float().numpy(), F, run(Xb, F, offset), offset)


def test_scales_of_rows_and_columns():
    print("[case] bf16 forms mixed scales", flush=True)
    rng = np.random.default_rng(5)
    shape, R = (40, 2, 31), 9
    X = rng.standard_normal(shape).astype(np.float32)
    X[3] *= np.float32(1e-35)
    X[7] = 0.0
    X[:, :, 5] *= np.float32(1e-36)
    F = [rng.uniform(0.5, 1.5, (n, R)).astype(np.float32) for n in shape]
    F[2][:, 4] *= np.float32(1e-33)
    F[1][:, 6] = 0.0
    Xb = bf16(X)
    got = run(Xb, F)
    check(Xb.float().numpy(), F, got)
    assert np.all(got[0][7] == 0.0) and np.all(got[0][:, 6] == 0.0)


@pytest.mark.parametrize("shape,offset", [((34, 2, 32), 1), ((35, 3, 33), 0), ((2, 32, 40), 0), ((2, 3, 40), 3)])
def test_infinities_and_nan(shape, offset):
    """As fp32 arithmetic gives them (see the fp32 kernel's test)."""
    print(f"[case] bf16 forms infinities {shape} offset={offset}", flush=True)
    rng = np.random.default_rng(7)
    R = 6
    X = rng.uniform(0.5, 1.0, shape).astype(np.float32)
    F = [rng.uniform(0.5, 1.0, (n, R)).astype(np.float32) for n in shape]
    F[1][0] *= -1
    X[0, 0, 3], X[1, 1, 2], X[1, 0, 1] = np.inf, -np.inf, np.nan
    F[2][5] = np.float32(3.4028235e38)
    X[:, :, 5] = 0.0
    Xb = bf16(X)
    got = run(Xb, F, offset)
    with np.errstate(all="ignore"):
        for m in range(3):
            if as_pair(shape, m, offset):
                continue
            ref = mttkrp64(Xb.float().numpy(), F, m)
            assert np.array_equal(np.isnan(got[m]), np.isnan(ref)), m
            big = np.isinf(ref)
            assert np.array_equal(got[m][big], ref[big].astype(np.float32)), m
