"""The vector kernels of the conjugate-gradient EEQ solves: the reciprocal product they frame
against its tensor form, and a whole solve against the assembled matrix, one and two columns,
row counts beside the chunk and workgroup edges, a column that is done before the other."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _system(n, seed=0, cell=True):
    from xnn_amd import eeq as E
    gen = torch.Generator().manual_seed(seed + n)
    side = 6.0 * max(n, 8) ** (1.0 / 3.0)
    pos = torch.rand(n, 3, dtype=torch.float64, generator=gen) * side
    c = torch.diag(torch.tensor([side, 1.1 * side, 0.9 * side], dtype=torch.float64)) if cell else None
    rad = 0.5 + torch.rand(n, dtype=torch.float64, generator=gen)
    diag = 2.0 + torch.rand(n, dtype=torch.float64, generator=gen) + math.sqrt(2.0 / math.pi) / rad
    alpha = E.ewald_alpha(24.0) if cell else 0.0
    args = [t if t is None else t.to(DEV) for t in (pos, c, rad, diag - 2 * alpha / math.sqrt(math.pi))]
    return E, gen, args, alpha, 24.0 if cell else math.inf


@pytest.mark.parametrize("n", [1, 31, 33, 255, 257, 8191, 8200])
@pytest.mark.parametrize("R", [1, 2])
def test_reciprocal_product(n, R):
    E, gen, (pos, cell, _, diag), alpha, _ = _system(n)
    m = E.reciprocal_half_set(cell, alpha)
    if n > 1000:
        m = m[:200].contiguous()              # the tensor form keeps (N, M) phases
    fr = E.FactorizedReciprocal(pos, cell, m, alpha)
    v = torch.randn(n, R, dtype=torch.float64, generator=gen).to(DEV)
    base = torch.randn(n, R, dtype=torch.float64, generator=gen).to(DEV)
    g, w = E.reciprocal_weights(m, cell, alpha)
    want = base + diag[:, None] * v + torch.stack([E._reciprocal_block(pos, g, w, v[:, k])
                                                   for k in range(R)], 1)
    eps = torch.finfo(torch.float64).eps
    scale = float(w.sum() * v.abs().sum() + base.abs().max())     # every phase at one
    torch.testing.assert_close(fr.add_to(base.clone(), v, diag), want, rtol=0, atol=64 * eps * scale)
    torch.testing.assert_close(fr.apply(v) + base + diag[:, None] * v, want, rtol=0, atol=64 * eps * scale)
    fr.table, fr.block = None, 3              # column blocks formed as they are needed
    torch.testing.assert_close(fr.add_to(base.clone(), v, diag), want, rtol=0, atol=64 * eps * scale)


@pytest.mark.parametrize("n,cell", [(1, False), (33, False), (33, True), (300, True), (1000, False)])
def test_solves_against_the_matrix(n, cell):
    E, gen, args, alpha, cutoff = _system(n, 5, cell)
    cg = E.IterativeEEQSystem(*args, alpha, cutoff)
    dense = E.LargeEEQSystem(*args, alpha, cutoff)
    b = torch.randn(n, 2, dtype=torch.float64, generator=gen).to(DEV)
    for cols, tols in ((b, [1e-11, 1e-2]), (b[:, :1].contiguous(), [1e-11])):
        tol = torch.tensor(tols, dtype=torch.float64, device=DEV)
        x = cg.conjugate_gradient(cols[cg.order], tol)
        out = torch.empty_like(x)
        out[cg.order] = x
        res = torch.linalg.vector_norm(cols - dense.A @ out, dim=0)
        # the recurrence's residual against the true one: rounding of the product
        assert (res <= tol + 1e-12 * float(dense.A.abs().max()) * torch.linalg.vector_norm(out, dim=0)).all()


@pytest.mark.parametrize("vectors", [1024, 1025, 1500])
@pytest.mark.parametrize("R", [1, 2])
def test_low_rank_parts_beyond_the_lds(monkeypatch, vectors, R):
    """2,048 columns of the preconditioner are the most that a workgroup's LDS takes."""
    E, gen, args, alpha, cutoff = _system(300, 5)
    monkeypatch.setattr(E, "LOW_K_VECTORS", vectors)
    cg = E.IterativeEEQSystem(*args, alpha, cutoff)
    assert cg.U.shape[1] == 2 * vectors
    dense = E.LargeEEQSystem(*args, alpha, cutoff)
    b = torch.randn(300, R, dtype=torch.float64, generator=gen).to(DEV)
    tol = torch.full((R,), 1e-11, dtype=torch.float64, device=DEV)
    out = torch.empty_like(b)
    out[cg.order] = cg.conjugate_gradient(b[cg.order], tol)
    res = torch.linalg.vector_norm(b - dense.A @ out, dim=0)
    assert (res <= tol + 1e-12 * float(dense.A.abs().max()) * torch.linalg.vector_norm(out, dim=0)).all()
