"""CP reconstruction of a vector whose tiles (128 x 128 elements, of which a vector fills one column) are more threads
than one launch takes: 2.2e9 rows at rank 1.  The result is the factor itself."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from tenrso_amd.kernels import cp_reconstruct  # noqa: E402


def test_more_tiles_than_a_launch():
    print("[case] reconstruction of 2200000000 elements, rank 1", flush=True)
    rows = 2_200_000_000
    if torch.cuda.mem_get_info()[0] < 24 << 30:
        pytest.skip("needs 24 GiB")
    f = torch.full((rows, 1), 1.5, device="cuda")
    stale = torch.zeros(rows, device="cuda")
    del stale  # (the result's memory)
    out = cp_reconstruct([f])
    assert float(out.min()) == 1.5 and float(out.max()) == 1.5
