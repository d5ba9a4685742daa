"""The stored real-space product of the EEQ conjugate-gradient regime
(``xnn_eeq_store_apply``) against the formed matrix, at the tiles' edges."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _system(n, seed=0):
    gen = torch.Generator().manual_seed(seed)
    box = 4.0 * max(n, 2) ** (1 / 3)
    cell = (torch.eye(3) * box + 0.05 * box * torch.rand((3, 3), generator=gen)).double()
    pos = (torch.rand((n, 3), generator=gen).double() @ cell).to(DEV)
    rad = (0.8 + torch.rand(n, generator=gen)).double().to(DEV)
    v = torch.randn((n, 2), generator=gen, dtype=torch.float64).to(DEV)
    return pos.contiguous(), cell.to(DEV), rad, v


@pytest.mark.parametrize("n", [1, 64, 127, 128, 129, 257, 1000])
@pytest.mark.parametrize("periodic", [True, False])
def test_stored_tiles_match_the_formed_matrix(n, periodic):
    from xnn_amd import eeq as E
    pos, cell, rad, v = _system(n)
    # a range longer than the small cells (own images) and shorter than the largest
    cutoff = 30.0 if periodic else float("inf")
    alpha = E.ewald_alpha(cutoff) if periodic else 0.0
    host = E._host_cell(cell) if periodic else None
    R = E.real_matrix(pos, cell if periodic else None, rad, alpha, cutoff)
    store = E.RealTiles.build(pos, host, rad, alpha, cutoff)
    # n products of magnitude |R| |v|, each rounded once, and kernel values to a few ulps
    bound = (n + 16) * 2.3e-16 * (R.abs() @ v.abs())
    for cols in (slice(0, 1), slice(0, 2)):
        got = store.apply(v[:, cols].contiguous())
        assert bool(((got - R @ v[:, cols]).abs() <= bound[:, cols] + 1e-300).all())
        assert torch.equal(store.apply(v[:, cols].contiguous()), got)


@pytest.mark.parametrize("n,periodic", [(129, False), (257, False), (1, False), (129, True)])
def test_every_tile_starts_within_the_values(n, periodic):
    """Also the last one where it is a single atom without an own image, which has none; a
    range of 10 bohr in a cell of 20 for the periodic case."""
    from xnn_amd import eeq as E
    pos, cell, rad, _ = _system(n)
    cutoff = 10.0 if periodic else float("inf")
    alpha = E.ewald_alpha(cutoff) if periodic else 0.0
    store = E.RealTiles.build(pos, E._host_cell(cell) if periodic else None, rad, alpha, cutoff)
    base = store._keep[-1]
    masks = store._keep[2].view(len(base), -1)
    assert bool((masks[-1] == 0).all())          # the case meant
    assert int(base.max()) < store.values.numel()


def test_far_tiles_are_left_out_and_the_fallback_agrees(monkeypatch):
    """Two clusters out of each other's reach: their tiles are not stored; without room for
    the tiles the regime evaluates its pairs at every product, to the same charges."""
    from xnn_amd import eeq as E
    gen = torch.Generator().manual_seed(4)
    n, cutoff = 512, 20.0
    cell = torch.diag(torch.tensor([30.0, 30.0, 400.0], dtype=torch.float64))
    pos = torch.rand((n, 3), generator=gen).double() * torch.tensor([30.0, 30.0, 30.0])
    pos[n // 2:, 2] += 200.0        # the most significant axis of the order
    pos, cell = pos.to(DEV), cell.to(DEV)
    rad = torch.full((n,), 1.2, dtype=torch.float64, device=DEV)
    diag = torch.full((n,), 3.0, dtype=torch.float64, device=DEV)
    x = torch.randn(n, generator=gen, dtype=torch.float64).to(DEV)
    alpha = E.ewald_alpha(cutoff)
    system = E.IterativeEEQSystem(pos, cell, rad, diag, alpha, cutoff)
    assert system.store is not None and system.store.tiles.n_tiles < 4 * 5 // 2
    zero = torch.zeros((), dtype=torch.float64, device=DEV)
    q, mu = system.solve_augmented(x, zero)
    monkeypatch.setattr(E, "STORE_BYTES", 0)
    free = E.IterativeEEQSystem(pos, cell, rad, diag, alpha, cutoff)
    assert free.store is None
    q2, mu2 = free.solve_augmented(x, zero)
    # both to a residual of 1e-12 |x|, the operator's smallest eigenvalue of order one
    assert float((q - q2).abs().max()) <= 2e-11 * float(x.norm())


def _charges(n, solver, seed=7):
    from xnn_amd import eeq as E
    pos, cell, rad, v = _system(n, seed)
    diag = torch.full((n,), 3.0, dtype=torch.float64, device=DEV)
    leaves = [pos.clone().requires_grad_(True), cell.clone().requires_grad_(True)]
    q = E.eeq_charges_large(leaves[0], leaves[1], rad, diag, v[:, 0].contiguous(), 0.0, 24.0,
                            solver=solver)
    return q, leaves, v[:, 1]


def test_values_are_given_back_between_the_solves(monkeypatch):
    """Neither the graph nor a second backward through it keeps the stored values."""
    from xnn_amd import eeq as E
    made = []
    form = E.IterativeEEQSystem._form_store
    monkeypatch.setattr(E.IterativeEEQSystem, "_form_store", lambda s: (made.append(s), form(s))[1])
    q, leaves, u = _charges(300, "cg")
    assert len(made) == 1 and made[0].store is None
    got = torch.autograd.grad([q], leaves, [u], retain_graph=True)
    assert len(made) == 2 and made[1] is made[0] and made[0].store is None
    again = torch.autograd.grad([q], leaves, [u])
    assert len(made) == 3 and made[0].store is None
    ref_q, ref_leaves, _ = _charges(300, "lu")
    want = torch.autograd.grad([ref_q], ref_leaves, [u])
    # both solved to 1e-12 of the right-hand side, eigenvalues of order one
    torch.testing.assert_close(q, ref_q, rtol=0, atol=1e-10)
    for a, b, c in zip(got, again, want):
        assert torch.equal(a, b)
        torch.testing.assert_close(a, c, rtol=0, atol=1e-9 * float(c.abs().max()))


def test_values_take_at_most_half_of_the_memory_left(monkeypatch):
    from xnn_amd import eeq as E
    pos, cell, rad, _ = _system(300)
    args = (pos, E._host_cell(cell), rad, E.ewald_alpha(30.0), 30.0)
    need = 8 * (E.RealTiles.build(*args).values.numel() - 1)
    for left, kept in ((2 * need, True), (2 * need - 2, False)):
        monkeypatch.setattr(E, "_device_left", lambda dev: left)
        assert (E.RealTiles.build(*args) is not None) == kept
