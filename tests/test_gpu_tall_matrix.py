"""MTTKRP of a matrix of so many rows that its tiles (32 rows by a window of 32 columns, 512 threads each) are more
threads than one launch takes (2^32 - 1): 54 million rows, five windows.  The factor's values are multiples of 2^-7 and
X is one, so every sum is exact."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from tenrso_amd import kernels  # noqa: E402


def test_more_tiles_than_a_launch():
    print("[case] bf16 mttkrp of 54000000 x 160, rank 1", flush=True)
    rows, cols = 54_000_000, 160
    if torch.cuda.mem_get_info()[0] < 24 << 30:
        pytest.skip("needs 24 GiB")
    X = torch.ones(rows, cols, dtype=torch.bfloat16, device="cuda")
    F = [torch.ones(rows, 1, device="cuda"), (torch.arange(cols, device="cuda", dtype=torch.float32) / 128)[:, None]]
    got = kernels.mttkrp_bf16(X, F, 0)
    want = float(cols * (cols - 1) / 2 / 128)
    assert got.shape == (rows, 1)
    assert float(got.min()) == want and float(got.max()) == want
