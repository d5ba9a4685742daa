"""The weight gradients of the fused linear message and of the node readout against float64
sums: empty rows, one atom, more rows than persistent waves, columns beside a tile's edge."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
EPS = torch.finfo(torch.float32).eps


@pytest.mark.parametrize("n,e,C,l_max,K", [(1, 0, 32, 1, 1), (1, 1, 64, 3, 8), (3, 200, 128, 2, 7),
                                           (5000, 9000, 64, 3, 8), (2100, 6000, 32, 1, 5),
                                           (40, 3000, 128, 3, 8)])
def test_linear_message_weight_gradient(n, e, C, l_max, K):
    import oracle.reference as R
    from xnn_amd.ops import sh_linear_message_sum_op
    gen = torch.Generator().manual_seed(n + e)
    vec, h = torch.randn(e, 3, generator=gen), torch.randn(e, K, generator=gen)
    W = torch.randn(K, C, generator=gen)
    dst = torch.randint(0, n, (e,), generator=gen).sort().values
    perm = torch.randperm(e, generator=gen)              # edge perm[j] is the j-th of the CSR
    ptr = torch.searchsorted(dst, torch.arange(n + 1)).to(torch.int32)
    G = torch.randn(n, C, (l_max + 1) ** 2, generator=gen)
    Wd = W.to(DEV).requires_grad_(True)
    A = sh_linear_message_sum_op(vec.to(DEV), h.to(DEV), Wd, ptr.to(DEV),
                                 perm.to(torch.int32).to(DEV), l_max, 1)
    (got,) = torch.autograd.grad([A], [Wd], [G.to(DEV)])
    Y = R.e3nn_sh(l_max, vec.double())[perm]
    d_phi = (G.double()[dst] * Y[:, None, :]).sum(-1)
    want = h.double()[perm].t() @ d_phi
    # per output the e (l_max + 1)^2 products of its sum, each to a few float32 roundings
    bound = 8 * EPS * (h.double()[perm].abs().t() @ (G.double()[dst].abs() * Y.abs()[:, None, :]).sum(-1))
    assert ((got.cpu().double() - want).abs() <= bound).all()


@pytest.mark.parametrize("n,F", [(1, 1), (31, 16), (33, 255), (64, 257), (3000, 1024)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("broadcast", [False, True])
def test_readout_weight_gradient(n, F, dtype, broadcast):
    from xnn_amd.ops import node_readout_op
    gen = torch.Generator().manual_seed(n + F)
    rows = torch.randn(n, F, generator=gen, dtype=dtype)
    w, bias = torch.randn(F, generator=gen, dtype=dtype), torch.zeros(3, dtype=dtype)
    g = torch.full((1,), -1.5, dtype=dtype).expand(n) if broadcast else torch.randn(n, generator=gen, dtype=dtype)
    wd = w.to(DEV).requires_grad_(True)
    E = node_readout_op(rows.to(DEV), wd, torch.zeros(n, dtype=torch.int64, device=DEV), bias.to(DEV))
    gd = g[:1].to(DEV).expand(n) if broadcast else g.to(DEV)
    (got,) = torch.autograd.grad([E], [wd], [gd])
    want = rows.double().t() @ g.double()
    eps = torch.finfo(dtype).eps
    # summed in float64 and rounded once
    bound = eps * want.abs() + (n + 1) * 2.3e-16 * (rows.double().abs().t() @ g.double().abs())
    assert ((got.cpu().double() - want).abs() <= bound).all()


def test_readout_weight_gradient_of_a_batch_of_cotangents():
    from xnn_amd.ops import node_readout_op
    gen = torch.Generator().manual_seed(1)
    rows, w, g = (torch.randn(*k, generator=gen).to(DEV) for k in ((50, 33), (33,), (4, 50)))
    w.requires_grad_(True)
    E = node_readout_op(rows, w, torch.zeros(50, dtype=torch.int64, device=DEV), torch.zeros(1, device=DEV))
    (got,) = torch.autograd.grad([E], [w], [g], is_grads_batched=True)
    bound = 52 * EPS * (g.double().abs() @ rows.double().abs())       # float32 products and sums
    assert ((got.double() - g.double() @ rows.double()).abs() <= bound).all()


@pytest.mark.parametrize("l_max", [1, 2, 3])
def test_linear_message_weight_gradient_of_a_misaligned_cotangent(l_max):
    """A cotangent that is a view one float into other memory is the same as any other."""
    from xnn_amd.ops import sh_linear_message_sum_op
    gen = torch.Generator().manual_seed(2)
    vec, h, W = (torch.randn(*k, generator=gen).to(DEV) for k in ((60, 3), (60, 8), (8, 32)))
    ptr = torch.arange(0, 61, 6, dtype=torch.int32, device=DEV)
    W.requires_grad_(True)
    A = sh_linear_message_sum_op(vec, h, W, ptr, None, l_max, 1)
    G = torch.randn(A.shape, generator=gen).to(DEV)
    view = torch.empty(A.numel() + 1, device=DEV)[1:].view_as(A).copy_(G)
    assert view.data_ptr() % 16
    want, got = (torch.autograd.grad([A], [W], [k], retain_graph=True)[0] for k in (G, view))
    assert torch.equal(got, want)
