"""``reciprocal_apply`` on the GPU (``xnn_eeq_recip``) against its tensor form in float64 on the
CPU: values, all four gradients, a gradient of a gradient, at the edges of its 256-wide tiles
and splits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("n,m", [(0, 5), (5, 0), (1, 1), (63, 257), (64, 256), (65, 255), (257, 63),
                                 (1000, 700), (1, 3000), (3000, 1)])
def test_values_and_gradients(n, m):
    from xnn_amd.eeq import _reciprocal_block, reciprocal_apply
    gen = torch.Generator().manual_seed(1000 * n + m)
    r = lambda *s: torch.randn(*s, dtype=torch.float64, generator=gen)
    host = [20.0 * r(n, 3), r(m, 3), r(m).abs(), r(n)]
    u = r(n)
    out = []
    for dev, fn in ((DEV, reciprocal_apply), ("cpu", _reciprocal_block)):
        args = [t.to(dev).requires_grad_(True) for t in host]
        y = fn(*args)
        grads = torch.autograd.grad([y], args, [u.to(dev)], allow_unused=True)
        fewer = torch.autograd.grad([fn(args[0], *[t.detach() for t in args[1:]])], args[:1], [u.to(dev)])
        out.append([t.detach().cpu() for t in (y, *grads, *fewer)])
    # a sum of n m terms of unit size times the largest factor beside them; phases up to 100
    # carry 100 eps, one part in eps each beyond
    tol = 200 * torch.finfo(torch.float64).eps * max(n * m, 1)
    for a, b in zip(*out):
        assert a.shape == b.shape
        torch.testing.assert_close(a, b, rtol=1e-11, atol=tol)


def test_gradient_of_the_gradient():
    from xnn_amd.eeq import _reciprocal_block, reciprocal_apply
    gen = torch.Generator().manual_seed(3)
    r = lambda *s: torch.randn(*s, dtype=torch.float64, generator=gen)
    host = [r(20, 3), r(30, 3), r(30).abs(), r(20)]
    res = []
    for dev, fn in ((DEV, reciprocal_apply), ("cpu", _reciprocal_block)):
        args = [t.to(dev).requires_grad_(True) for t in host]
        first = torch.autograd.grad([fn(*args).sin().sum()], args, create_graph=True)
        second = torch.autograd.grad([sum((t * t).sum() for t in first)], args)
        res.append([t.detach().cpu() for t in second])
    for a, b in zip(*res):
        torch.testing.assert_close(a, b, rtol=1e-10, atol=1e-10 * float(b.abs().max()))


def test_forward_mode_and_batched_gradients():
    """A directional derivative (dual numbers and functional) is the gradient times the
    direction, also over a batch of vectors; a batch of cotangents is one after another."""
    from torch.autograd import forward_ad as fw
    from xnn_amd.eeq import reciprocal_apply
    gen = torch.Generator().manual_seed(4)
    r = lambda *s: torch.randn(*s, dtype=torch.float64, generator=gen).to(DEV)
    pos, g, w, v, u, t = r(20, 3), r(30, 3), r(30).abs(), r(20), r(3, 20), r(20, 3)
    leaf = pos.clone().requires_grad_(True)
    out = reciprocal_apply(leaf, g, w, v)
    rows = torch.stack([torch.autograd.grad(out, leaf, k, retain_graph=True)[0] for k in u])
    want = torch.einsum("bij,ij->b", rows, t)
    tol = dict(rtol=0, atol=1e-12 * float(rows.abs().sum(0).max()) * 60)
    with fw.dual_level():
        tangent = fw.unpack_dual(reciprocal_apply(fw.make_dual(pos, t), g, w, v)).tangent
    torch.testing.assert_close(u @ tangent, want, **tol)
    f = lambda p: reciprocal_apply(p, g, w, v)
    torch.testing.assert_close(u @ torch.func.jvp(f, (pos,), (t,))[1], want, **tol)
    torch.testing.assert_close(torch.func.vmap(lambda k: reciprocal_apply(pos, g, w, k))(u),
                               torch.stack([reciprocal_apply(pos, g, w, k) for k in u]), **tol)
    (got,) = torch.autograd.grad(out, leaf, u, is_grads_batched=True)
    torch.testing.assert_close(got, rows, **tol)
