"""The MTTKRP on bf16 parts where some values lie near the lower end of the exponent range: in every tile form
(window fully or partly filled, rank tiles of 1 to 8, all modes in one launch, the bf16 last mode), against FP64.

TINY is 2^-121 with bits down to 2^-134, below the last bit of any bf16 value (2^-133): as a sum of bf16 parts it
is off by 2^-13 of itself, wherever it stands, and always in the same direction.  All other values are positive, of
magnitude 0.5 to 2, so every product with it is a normal fp32 number.

Tolerance: that of the fp32 kernel's tests, (J + 8) 2^-23 sum |x kr| per element; J is below 1000, so a lost part
of TINY exceeds it.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from test_gpu_bf16_forms import bf16  # noqa: E402
from test_gpu_mttkrp_split import check, mttkrp64, run  # noqa: E402

from tenrso_amd import kernels  # noqa: E402

TINY = np.float32(4097.4375 * 2.0 ** -133)


def positive(shape, R):
    rng = np.random.default_rng(sum(shape) + R)
    X = rng.uniform(0.5, 2.0, shape).astype(np.float32)
    return X, [rng.uniform(0.5, 2.0, (n, R)).astype(np.float32) for n in shape]


def check_all(X, F):
    check(X, F, run(X, F))
    got = kernels.mttkrp_all_modes(torch.from_numpy(X).cuda(), [torch.from_numpy(f).cuda() for f in F])
    check(X, F, [g.cpu().numpy() for g in got])
    # bf16: the last mode takes exact parts of its fastest factor too
    Xb, last = bf16(X), X.ndim - 1
    got = kernels.mttkrp_bf16(Xb.cuda(), [torch.from_numpy(f).cuda() for f in F], last).cpu().numpy()
    X32, J = Xb.float().numpy(), X.size // X.shape[-1]
    lim = (J + 8) * 2.0 ** -23 * mttkrp64(X32, F, last, mag=True) + 1e-44
    assert np.all(np.abs(got - mttkrp64(X32, F, last)) <= lim)


def check_column(shape, R, col):
    print(f"[case] small column {shape} R={R} column {col}", flush=True)
    for k in (-1, -2):  # the fastest factor of every mode but the last, and that of the last
        X, F = positive(shape, R)
        F[k][:, col] = TINY
        check_all(X, F)


@pytest.mark.parametrize("shape,R,col", [((34, 3, 33), 65, 64), ((34, 4, 35), 100, 70), ((33, 5, 40), 128, 127),
                                         ((5, 6, 128), 128, 64)])
def test_small_column_past_64(shape, R, col):
    check_column(shape, R, col)


@pytest.mark.parametrize("shape,R,col", [((5, 2, 32), 9, 4), ((6, 32, 32), 8, 5), ((3, 64, 64), 8, 3), ((4, 96, 64), 40, 37),
                                         ((3, 5, 160), 64, 60), ((3, 4, 32, 96), 20, 17), ((34, 4, 32), 100, 70)])
def test_small_column_beside_an_unfilled_window(shape, R, col):
    check_column(shape, R, col)


@pytest.mark.parametrize("shape,R", [((5, 2, 32), 9), ((35, 3, 33), 20), ((6, 32, 64), 64), ((6, 4, 32), 100), ((3, 4, 5, 64), 40)])
def test_small_entries_that_decide_a_result(shape, R):
    """Small entries of a row or column whose other entries are not, where those others meet exact zeros."""
    print(f"[case] small entries {shape} R={R}", flush=True)
    X, F = positive(shape, R)
    X[..., 5] = TINY
    F[-1][:, 3] = 0.0
    F[-1][5, 3] = 1.75
    check_all(X, F)
    X, F = positive(shape, R)
    X[..., 7] = 0.0
    X[1, ..., 7] = 1.5
    X[1, ..., :7] = 0.0
    X[1, ..., 8:] = 0.0
    F[-1][7, 3] = TINY
    check_all(X, F)


def test_products_that_only_the_third_factor_makes_normal():
    print("[case] small products", flush=True)
    X, F = positive((40, 3, 32), 20)
    X *= np.float32(2.0 ** -70)
    F[2] *= np.float32(2.0 ** -70)
    F[1] *= np.float32(2.0 ** 60)
    check_all(X, F)
    X, F = positive((40, 32, 33), 70)
    X *= np.float32(2.0 ** -70)
    F[1] *= np.float32(2.0 ** -70)
    F[0] *= np.float32(2.0 ** 60)
    F[2] *= np.float32(2.0 ** 60)
    check_all(X, F)


@pytest.mark.parametrize("shape,R", [((70, 33, 130), 16), ((64, 40, 256), 33), ((33, 70, 97), 64), ((9000, 2, 20), 8), ((2, 20, 9001), 24),
                                     ((40, 64, 66), 128), ((35, 3, 4, 67), 100), ((20, 9, 11, 32), 40)])
def test_tiles_formed_again(shape, R):
    """A small value, an infinity and a NaN in many tiles: every other result keeps its tolerance."""
    print(f"[case] tiles again {shape} R={R}", flush=True)
    X, F = positive(shape, R)
    X.reshape(-1)[::97] = TINY
    check_all(X, F)
    X.reshape(-1)[0] = np.inf
    X.reshape(-1)[X.size // 2] = np.nan
    got = kernels.mttkrp_all_modes(torch.from_numpy(X).cuda(), [torch.from_numpy(f).cuda() for f in F])
    one = run(X, F)
    for m in range(X.ndim):
        with np.errstate(invalid="ignore"):
            ref = mttkrp64(X, F, m)
        fin = np.isfinite(ref)
        lim = (X.size // X.shape[m] + 8) * 2.0 ** -23 * np.abs(ref)
        for g in (got[m].cpu().numpy(), one[m]):
            assert np.array_equal(np.isnan(g), np.isnan(ref)) and np.array_equal(np.isposinf(g), np.isposinf(ref)), m
            assert np.all(np.abs(g[fin] - ref[fin]) <= lim[fin]), m


def test_a_nan_costs_a_second_pass():
    """Forming a tile again takes the order of the launch's time, not that of a serial loop (25 to 50 times it)."""
    print("[case] time with a NaN", flush=True)
    X = torch.ones((256, 256, 256), device="cuda")
    F = [torch.ones((256, 64), device="cuda") for _ in range(3)]

    def best():
        ms = []
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(10):
                kernels.mttkrp(X, F, 1)
            b.record()
            b.synchronize()
            ms.append(a.elapsed_time(b))
        return min(ms)

    ordinary = best()
    X[3, 4, 5] = float("nan")
    assert best() <= 8 * ordinary
