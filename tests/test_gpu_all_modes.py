"""mttkrp_all_modes in one call, and where the kernel allows it in one launch, against FP64: the tolerance of the
fp32 kernel's own tests, (J + 8) 2^-23 sum |x kr| per element."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from test_gpu_mttkrp_split import check  # noqa: E402

from tenrso_amd import kernels  # noqa: E402


# (2, 2, 2, 2, 2) and (3, 2, 4, 2) rank 40: more Khatri-Rao elements than the batch takes; eight modes: the most;
# rank 130, a last mode of one row, no elements, no columns: a launch a mode or none; an offset: unaligned rows
@pytest.mark.parametrize("shape,R", [((5, 7), 3), ((64, 32), 40), ((33, 1, 31), 8), ((250, 34, 66), 64), ((40, 33, 64), 130),
                                     ((12, 20, 9, 32), 16), ((3, 2, 4, 2), 40), ((2, 2, 2, 2, 2), 5), ((4, 8, 6, 7, 5), 3),
                                     ((2, 3, 2, 2, 3, 2, 2, 3), 2), ((4, 0, 3), 2), ((4, 3, 2), 0), ((9, 8, 1), 5),
                                     ((64, 64, 64), 32), ((100, 2, 64), 17), ((16, 200, 32), 64), ((300, 96, 33), 7),
                                     ((32, 3, 7, 9001), 4), ((8, 8, 32, 2), 12)])
def test_all_modes(shape, R):
    print(f"[case] all modes {shape} R={R}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(sum(shape) + R)
    X = torch.randn(shape, generator=g, device="cuda")
    F = [torch.randn((n, R), generator=g, device="cuda") for n in shape]
    flat = torch.empty(X.numel() + 1, device="cuda")
    flat[1:] = X.reshape(-1)
    for T in (X, X.transpose(0, 1).contiguous().transpose(0, 1), flat[1:].view(shape)):
        got = kernels.mttkrp_all_modes(T, F)
        assert [tuple(o.shape) for o in got] == [(n, R) for n in shape]
        if X.numel() * R:
            check(X.cpu().numpy(), [f.cpu().numpy() for f in F], [o.cpu().numpy() for o in got])


def test_infinities_and_small_values():
    """One mode's tiles in plain fp32 arithmetic, whatever the others need."""
    X = torch.randn((40, 33, 35), device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    F = [torch.rand((n, 6), device="cuda") + 0.5 for n in X.shape]
    X[3, 4, 5] = float("inf")
    X[7] *= 1e-35
    for m, o in enumerate(kernels.mttkrp_all_modes(X, F)):
        row = (3, 4, 5)[m]
        assert bool(torch.isposinf(o[row]).all()) and bool(torch.isfinite(o[[i for i in range(o.shape[0]) if i != row]]).all())
        if m == 0:
            want = torch.einsum("jk,jr,kr->r", X[7].double(), F[1].double(), F[2].double())
            mag = torch.einsum("jk,jr,kr->r", X[7].double().abs(), F[1].double(), F[2].double())
            assert bool(((o[7].double() - want).abs() <= (33 * 35 + 8) * 2.0 ** -23 * mag).all())


def test_refused_as_one_by_one():
    X = torch.zeros((4, 3, 2), device="cuda")
    F = [torch.zeros((n, 2), device="cuda") for n in (4, 3, 2)]
    for bad in (F[:2], F[:2] + [torch.zeros((2, 3), device="cuda")], [F[1], F[0], F[2]]):
        with pytest.raises(ValueError) as one:
            kernels.mttkrp(X, bad, 0)
        with pytest.raises(ValueError) as every:
            kernels.mttkrp_all_modes(X, bad)
        assert str(one.value) == str(every.value)
    with pytest.raises(TypeError):
        kernels.mttkrp_all_modes(X.double(), F)
    got = kernels.mttkrp_all_modes(X, [f.double().cpu().numpy() for f in F])  # converted, as by mttkrp
    assert all(np.all(o.cpu().numpy() == 0.0) for o in got)
