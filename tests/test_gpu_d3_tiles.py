"""The D3 pair and coordination tiles at the edges of their 64-atom tiles: the two-body term
against the general kernel over directed pairs, the counts against the oracle."""
import os

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


def _inputs(counts, periodic, seed=5):
    rng = np.random.default_rng(seed)
    z = rng.choice([1, 6, 7, 8], size=sum(counts))
    pos, cells = [], []
    for n in counts:
        side = max(6.0, (n / 0.08) ** (1 / 3))
        cell = np.diag([side, side * 1.1, side * 0.95]) + rng.normal(scale=0.2, size=(3, 3))
        pos.append(rng.uniform(-0.3, 1.3, (n, 3)) @ cell)
        cells.append(cell)
    return z, np.concatenate(pos), np.stack(cells) if periodic else None


@pytest.mark.parametrize("counts", [[1], [63], [64], [65], [200], [5, 130, 64]])
@pytest.mark.parametrize("periodic", [True, False])
def test_tiles_match_the_general_kernel(counts, periodic):
    import xnn_amd.dispersion as XD
    from xnn_amd.dispersion import load_d3_tables
    tables = load_d3_tables(os.path.join(GOLDEN, "d3_tables_hcnoar.npz"))
    z, pos, cell = _inputs(counts, periodic)
    results = []
    for tiles in (True, False):
        model = XD.DFTD3(tables, cutoff_pair=11.0, cutoff_cn=9.0, switch_width_pair=1.5).to(DEV)
        assert model._pair_tiles
        model._pair_tiles = tiles
        p = torch.tensor(pos, device=DEV, requires_grad=True)
        c = None if cell is None else torch.tensor(cell, device=DEV, requires_grad=True)
        pbc = None if cell is None else torch.ones((len(counts), 3), dtype=torch.bool)
        leaves = [p] if c is None else [p, c]
        out = model.evaluate(torch.tensor(z, device=DEV), p, c, pbc, torch.tensor(counts))
        seed = torch.linspace(-1.0, 2.0, len(z), dtype=torch.float64, device=DEV)
        both = [out["node_energy"].detach()]
        both += torch.autograd.grad((out["node_energy"] * seed).sum(), leaves)
        fused = model.evaluate(torch.tensor(z, device=DEV), p, c, pbc, torch.tensor(counts),
                               fused_pair=True)
        both += [fused["node_energy"].detach()] + list(torch.autograd.grad(fused["energy"].sum(), leaves))
        results.append((both, out["coordination_numbers"].detach()))
    energy = float(results[1][0][0].abs().max())
    for a, b in zip(results[0][0], results[1][0]):
        # sums of a few thousand terms of either sign in another order (a lone atom's forces
        # cancel to nothing: the terms are of the energy's size per Angstrom)
        torch.testing.assert_close(a, b, rtol=0, atol=2e-13 * (float(b.abs().max()) + energy))
    import oracle.d3 as D3
    from oracle.d4 import BOHR, edge_vectors_au, pair_images
    s0 = 0
    for k, n in enumerate(counts):
        one = slice(s0, s0 + n)
        c = None if cell is None else cell[k]
        dst, src, sh = pair_images(pos[one], c, 11.0)     # the image range of the longer cutoff
        r = torch.linalg.norm(edge_vectors_au(torch.tensor(pos[one]),
                                              None if c is None else torch.tensor(c), dst, src, sh), dim=-1)
        ref = D3.coordination_numbers(D3.species_of(tables, z[one]), dst, src, r, tables, 9.0 / BOHR, n)
        np.testing.assert_allclose(results[0][1][one].cpu(), ref, rtol=1e-12, atol=1e-13)
        s0 += n


@pytest.mark.parametrize("counts", [[70], [5, 130]])
@pytest.mark.parametrize("periodic", [True, False])
def test_a_shift_of_all_atoms_changes_nothing(counts, periodic):
    """A pair vector is rounded to its own length, wherever the structure lies: positions on a
    grid of 2^-20 Angstrom, so that a shift by 2^20 Angstrom changes no difference of two."""
    import xnn_amd.dispersion as XD
    tables = XD.load_d3_tables(os.path.join(GOLDEN, "d3_tables_hcnoar.npz"))
    z, pos, cell = _inputs(counts, periodic)
    pos = np.round(pos * 2.0 ** 20) / 2.0 ** 20
    model = XD.DFTD3(tables, cutoff_pair=11.0, cutoff_cn=9.0, switch_width_pair=1.5, s9=0.0).to(DEV)
    results = []
    for shift in (0.0, 2.0 ** 20):
        p = torch.tensor(pos + shift, device=DEV, requires_grad=True)
        c = None if cell is None else torch.tensor(cell, device=DEV, requires_grad=True)
        pbc = None if cell is None else torch.ones((len(counts), 3), dtype=torch.bool)
        out = model.evaluate(torch.tensor(z, device=DEV), p, c, pbc, torch.tensor(counts))
        grads = torch.autograd.grad(out["energy"].sum(), [p] if c is None else [p, c])
        results.append([out["coordination_numbers"].detach(), out["node_energy"].detach(), *grads])
    energy = float(results[0][1].abs().max())
    for a, b in zip(*results):
        # the same terms in another order: sums of a few thousand, as above
        torch.testing.assert_close(b, a, rtol=0, atol=2e-13 * (float(a.abs().max()) + energy))


def test_an_unsymmetric_table_takes_the_general_kernel():
    import xnn_amd.dispersion as XD
    tables = dict(XD.load_d3_tables(os.path.join(GOLDEN, "d3_tables_hcnoar.npz")))
    tables["c6ref"] = tables["c6ref"].copy()
    tables["c6ref"][0, 1, 0, 1] *= 1.01
    assert not XD.DFTD3(tables)._pair_tiles
    assert not XD.DFTD3(XD.load_d3_tables(os.path.join(GOLDEN, "d3_tables_hcnoar.npz")),
                        damping="zero")._pair_tiles


@pytest.mark.parametrize("damping", ["zero", "mzero", "op"])
def test_a_damping_set_afterwards_is_the_one_used(damping):
    import xnn_amd.dispersion as XD
    tables = XD.load_d3_tables(os.path.join(GOLDEN, "d3_tables_hcnoar.npz"))
    z, pos, _ = _inputs([30], False)
    args = (torch.tensor(z, device=DEV), torch.tensor(pos, device=DEV), None, None, torch.tensor([30]))
    later, model = XD.DFTD3(tables).to(DEV), XD.DFTD3(tables, damping=damping).to(DEV)
    later.damping = damping
    later.s6, later.s8, later.a1, later.a2 = model.s6, model.s8, model.a1, model.a2
    later.rs6, later.rs8, later.alp, later.bet = model.rs6, model.rs8, model.alp, model.bet
    assert torch.equal(later.evaluate(*args)["node_energy"], model.evaluate(*args)["node_energy"])
