"""mttkrp_all_modes in one call: the results of the modes one by one, bit for bit (the same kernels with the
same split of the work; only the reductions share a launch)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from tenrso_amd import kernels  # noqa: E402


# (2, 2, 2, 2, 2) and (3, 2, 4, 2) rank 40: more Khatri-Rao elements than the batch takes; eight modes: the most
@pytest.mark.parametrize("shape,R", [((5, 7), 3), ((64, 32), 40), ((33, 1, 31), 8), ((250, 34, 66), 64), ((40, 33, 64), 130),
                                     ((12, 20, 9, 32), 16), ((3, 2, 4, 2), 40), ((2, 2, 2, 2, 2), 5), ((4, 8, 6, 7, 5), 3),
                                     ((2, 3, 2, 2, 3, 2, 2, 3), 2), ((4, 0, 3), 2), ((4, 3, 2), 0)])
def test_as_one_by_one(shape, R):
    print(f"[case] all modes {shape} R={R}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(sum(shape) + R)
    X = torch.randn(shape, generator=g, device="cuda")
    F = [torch.randn((n, R), generator=g, device="cuda") for n in shape]
    for T in (X, X.transpose(0, 1).contiguous().transpose(0, 1)):
        got = kernels.mttkrp_all_modes(T, F)
        assert [tuple(o.shape) for o in got] == [(n, R) for n in shape]
        for m, o in enumerate(got):
            assert torch.equal(o, kernels.mttkrp(X, F, m)), m


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
