"""The three-body term's edge vectors (``dispersion._triple_vectors``) and their derivatives
against the plain tensor formulation, over the batches it accepts."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("case", ["molecules", "cell", "mixed", "far"])
def test_triple_vectors_match_the_tensor_form(case):
    from xnn_amd import dispersion as XD
    gen = torch.Generator().manual_seed(2)
    counts = {"molecules": [7, 0, 12, 1], "cell": [9], "mixed": [6, 5, 8], "far": [9]}[case]
    n = sum(counts)
    pos = (4.0 * torch.rand((n, 3), generator=gen, dtype=torch.float64)).to(DEV)
    cell = pbc = None
    if case != "molecules":
        cell = (torch.eye(3) * 6.0 + 0.3 * torch.rand((len(counts), 3, 3), generator=gen)).double()
        pbc = torch.ones((len(counts), 3), dtype=torch.bool)
        if case == "mixed":
            cell[1], pbc[1] = 0.0, False
        if case == "far":                     # an atom 600 cells away: the shifts leave 10 bits
            pos[4] += 600.0 * cell[0, 0].to(DEV)
        cell = cell.to(DEV)
    leaves = [t.clone().requires_grad_(True) for t in (pos, cell) if t is not None]
    ei, vec = XD.triple_graph(leaves[0], leaves[1] if cell is not None else None, pbc, counts, 5.0)
    g = torch.randn(vec.shape, generator=gen, dtype=torch.float64).to(DEV)
    got = torch.autograd.grad([vec], leaves, [g])
    # the reference: every structure's own list, in the list's order
    from xnn_amd.data import build_neighbor_list
    ref_leaves = [t.clone().requires_grad_(True) for t in (pos, cell) if t is not None]
    parts, edges, s0 = [], [], 0
    for b, k in enumerate(counts):
        p = ref_leaves[0][s0:s0 + k]
        periodic = cell is not None and bool(pbc[b].any())
        e, h = build_neighbor_list(p.detach(), 5.0, cell[b] if periodic else None,
                                   pbc[b] if periodic else None)
        v = p[e[1]] - p[e[0]]
        parts.append((v + h.double() @ ref_leaves[1][b] if periodic else v) / XD.BOHR)
        edges.append(e + s0)
        s0 += k
    ref_v, ref_e = torch.cat(parts), torch.cat(edges, 1)
    # the batched list may order a receiver's senders differently (no two images here)
    if case == "molecules":
        a, b = (torch.argsort(e[1] * n + e[0]) for e in (ei, ref_e))
        inverse = torch.empty_like(b)
        inverse[b] = a
        assert torch.equal(ei[:, inverse], ref_e)
        ref_g = g[inverse]
        vec = vec[inverse]
    else:
        assert torch.equal(ei, ref_e)
        ref_g = g
    # one rounding more or less in each term of order 10 (far: 3600) bohr
    tol = 1e-14 * float(ref_leaves[0].detach().abs().max())
    torch.testing.assert_close(vec, ref_v, rtol=0, atol=8 * tol)
    for a, b in zip(got, torch.autograd.grad([ref_v], ref_leaves, [ref_g])):
        torch.testing.assert_close(a, b, rtol=0, atol=1e-13 * float(b.abs().max()))


@pytest.mark.parametrize("periodic", [False, True])
def test_a_shift_of_all_atoms_changes_no_vector(periodic):
    """Positions on a grid of 2^-20 Angstrom in a cell of 8: a shift by 2^20 Angstrom (whole
    cells) changes no difference of two positions, so every bit stays."""
    from xnn_amd import dispersion as XD
    gen = torch.Generator().manual_seed(3)
    counts = [20] if periodic else [12, 8]
    pos = (torch.randint(0, 1 << 23, (20, 3), generator=gen).double() / 2.0 ** 20).to(DEV)
    cell = 8.0 * torch.eye(3, dtype=torch.float64, device=DEV)[None] if periodic else None
    pbc = torch.ones((1, 3), dtype=torch.bool) if periodic else None
    (e0, v0), (e1, v1) = (XD.triple_graph(pos + s, cell, pbc, counts, 5.0) for s in (0.0, 2.0 ** 20))
    assert e0.shape[1] > 20 and torch.equal(e0, e1) and torch.equal(v0, v1)


def test_other_refusals_of_the_plan_are_not_hidden():
    """Only shifts beyond the plan's 10 bits go on in the tensor form (``far`` above)."""
    from xnn_amd import dispersion as XD
    pos = torch.rand((5, 3), dtype=torch.float64, device=DEV)
    ei = torch.tensor([[0, 1], [1, 0]], device=DEV)
    with pytest.raises(ValueError, match="sums to 6"):
        XD._triple_vectors(pos, None, ei, torch.zeros((2, 3), dtype=torch.long, device=DEV), [6])


def test_vectors_have_a_tangent():
    """Forward-mode derivatives: the vectors are linear in the positions and the cell."""
    from torch.autograd import forward_ad as fw
    from xnn_amd import dispersion as XD
    gen = torch.Generator().manual_seed(6)
    pos = (4.0 * torch.rand((9, 3), generator=gen, dtype=torch.float64)).to(DEV)
    cell = (6.0 * torch.eye(3, dtype=torch.float64))[None].to(DEV)
    with fw.dual_level():
        _, v = XD.triple_graph(fw.make_dual(pos, pos), fw.make_dual(cell, cell), None, [9], 5.0)
        value, tangent = fw.unpack_dual(v)
    torch.testing.assert_close(tangent, value, rtol=0, atol=1e-14 * float(value.abs().max()))
