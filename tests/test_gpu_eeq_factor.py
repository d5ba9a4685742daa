"""``xnn_eeq_cholesky``: the factor and the diagonal blocks' inverses against LAPACK's at the
edges of its 16, 32, 64 and 128 wide tiles, and the first pivot that is not positive in every
part of a block."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 63, 127, 128, 129, 144, 191, 192, 193, 255, 257, 641])
def test_factor_and_inverses(n):
    from xnn_amd.eeq import _cholesky
    g = torch.Generator().manual_seed(n)
    M = torch.randn((n, n), dtype=torch.float64, generator=g)
    A = M @ M.T + n * torch.eye(n, dtype=torch.float64)
    L, info, inv = _cholesky(A.to(DEV), keep_inverses=True)
    assert int(info) == 0
    ref = torch.linalg.cholesky(A)
    # condition numbers below 6: a few units in the last place per term of the longest sum
    tol = 4 * n * torch.finfo(torch.float64).eps
    torch.testing.assert_close(L.cpu(), ref, rtol=0, atol=tol * float(ref.abs().max()))
    for k in range(0, n, 128):
        b = min(128, n - k)
        got = inv[k * 128:k * 128 + b * b].view(b, b).cpu()
        want = torch.linalg.inv(ref[k:k + b, k:k + b])
        torch.testing.assert_close(got, want, rtol=0, atol=tol * float(want.abs().max()))


@pytest.mark.parametrize("at", [0, 1, 15, 16, 100, 127, 128, 143, 200, 299])
@pytest.mark.parametrize("value", [-1.0, 0.0, float("nan"), float("inf")])
def test_first_bad_pivot(at, value):
    from xnn_amd.eeq import _cholesky
    A = torch.eye(300, dtype=torch.float64) * 2.0
    A[at, at] = value
    A[299, 299] = min(float(A[299, 299]), -1.0) if value == value else -1.0
    _, info = _cholesky(A.to(DEV))
    assert int(info) == at + 1
