"""Repeated-atom triangles of cells narrower than the three-body cutoff (own images, several
images of one neighbor, rows over one 64-edge tile) against the oracle's walk of every corner,
with different factors on the two sides of a pair C6 that is symmetric."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("n,cell,cutoff", [(1, 4.0, 9.0), (2, 5.0, 11.0), (5, 6.0, 10.0),
                                           (12, 9.0, 9.5)])
@pytest.mark.parametrize("width,alp3,k", [(0.0, 16.0 / 3.0, 23), (1.5, 16.0 / 3.0, 28), (0.0, 4.0, 5)])
def test_repeated_triangles_match_the_oracle(n, cell, cutoff, width, alp3, k):
    import oracle.d4 as D
    import xnn_amd.dispersion as XD
    from oracle.d4 import pair_images
    rng = np.random.default_rng(n)
    box = np.diag([cell, cell * 1.1, cell * 0.95]) + rng.normal(scale=0.1, size=(3, 3))
    pos = rng.uniform(0, 1, (n, 3)) @ box
    dst, src, sh = pair_images(pos, box, cutoff)
    order = rng.permutation(len(dst))
    ei, sh = torch.tensor(np.stack([src, dst])[:, order]), torch.tensor(sh[order]).double()
    factors = torch.tensor(rng.uniform(0.5, 2.0, (n, k)))
    mix = torch.tensor(rng.uniform(0.1, 1.0, (k, k)))
    mix = mix + mix.T                                  # <f S, f> is symmetric
    species = torch.tensor(rng.integers(0, 3, n))
    table = torch.tensor(rng.uniform(1.5, 3.0, (3, 3)))
    table = table + table.T
    go = torch.tensor(rng.normal(size=n))
    seeds = []
    for gpu in (True, False):
        # through positions and cell: a distinct triangle's gradient may sit on any corner's edges
        p = torch.tensor(pos, requires_grad=True)
        c = torch.tensor(box, requires_grad=True)
        v = p[ei[1]] - p[ei[0]] + sh @ c
        f = factors.clone().requires_grad_(True)
        if gpu:
            consts = XD.ATMConstants(species.int().to(DEV), table.to(DEV), 1.0, alp3, cutoff, width)
            vg, fg = v.to(DEV), f.to(DEV)
            e = XD.atm_energy(ei.to(DEV), vg, fg @ mix.to(DEV), fg, consts, n).cpu()
        else:
            e = D.atm_edges(ei, v, f @ mix, f, species, table, 1.0, alp3, cutoff, width, n)
        seeds.append((e.detach(), *torch.autograd.grad((e * go).sum(), [p, c, f])))
    scale = float(seeds[1][2].abs().max())             # the cell's: a lone atom's forces cancel
    for k, (a, b) in enumerate(zip(*seeds)):
        # some 1e5 terms of either sign, each to a few ulps
        atol = 1e-12 * (scale if k == 1 else float(b.abs().max()))
        torch.testing.assert_close(a, b, rtol=0, atol=atol)
