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


@pytest.mark.parametrize("k0,b", [(0, 128), (128, 128), (256, 44), (7, 1), (100, 77)])
def test_one_block(k0, b):
    """``xnn_eeq_cholesky_block`` by itself, anywhere in the matrix, and nothing beside it."""
    from xnn_amd import _lib
    g = torch.Generator().manual_seed(b)
    M = torch.randn((300, 300), dtype=torch.float64, generator=g)
    A = M @ M.T + 300 * torch.eye(300, dtype=torch.float64)
    got, inv = A.to(DEV), torch.empty(b, b, dtype=torch.float64, device=DEV)
    info = torch.zeros(1, dtype=torch.int32, device=DEV)
    _lib.call("xnn_eeq_cholesky_block", _lib.ptr(got), 300, k0, b, _lib.ptr(inv), _lib.ptr(info),
              _lib.stream(got.device))
    want = torch.linalg.cholesky(A[k0:k0 + b, k0:k0 + b])
    tol = 4 * b * torch.finfo(torch.float64).eps             # as above
    block = got.cpu()[k0:k0 + b, k0:k0 + b]
    torch.testing.assert_close(block, want, rtol=0, atol=tol * float(want.abs().max()))
    inverse = torch.linalg.inv(want)
    torch.testing.assert_close(inv.cpu(), inverse, rtol=0, atol=tol * float(inverse.abs().max()))
    rest = got.cpu()
    rest[k0:k0 + b, k0:k0 + b] = A[k0:k0 + b, k0:k0 + b]
    assert int(info) == 0 and torch.equal(rest, A)
