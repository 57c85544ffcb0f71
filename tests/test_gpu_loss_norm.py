"""||X||^2 inside the CP loss, summed by the MTTKRP kernel that reads X: every element once, whatever the
tile edges, the load form and the window.  With zero factors the loss is half of it.

Tolerance: FP64 sums of exact squares, n roundings of at most 2^-53: n 2^-53.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from tenrso_amd.ad import cp_loss_and_grad  # noqa: E402


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("shape,R", [((2, 3), 2), ((33, 31), 16), ((64, 32, 64), 8), ((5, 7, 1), 3), ((3, 5, 33), 20),
                                     ((31, 130, 35), 64), ((4, 6, 5, 7), 4), ((9, 31, 3, 64), 32), ((33, 8, 40, 3), 17),
                                     ((3, 2, 4, 3, 5), 6)])
def test_loss_of_zero_factors_is_half_the_norm(shape, R, offset):
    print(f"[case] loss norm {shape} R={R} offset={offset}", flush=True)
    rng = np.random.default_rng(sum(shape))
    X = rng.standard_normal(shape).astype(np.float32)
    flat = torch.empty(X.size + offset, device="cuda")
    flat[offset:] = torch.from_numpy(X).cuda().reshape(-1)
    F = [torch.zeros((n, R), device="cuda") for n in shape]
    want = 0.5 * float(np.sum(X.astype(np.float64) ** 2))
    for with_grad in (True, False):
        loss, _ = cp_loss_and_grad(flat[offset:].view(shape), F, with_grad)
        assert abs(loss - want) <= X.size * 2.0 ** -53 * want
