"""``xnn_eeq_real_grad_pairs`` (unordered 64 x 64 tiles) against the directed kernel: edges of
tiles, several images a pair, an atom's own images, molecules, no cell gradient wanted."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 129, 300])
@pytest.mark.parametrize("kind", ["narrow", "wide", "molecule", "no_cell_gradient"])
def test_pairs_match_the_directed_sum(n, kind):
    from xnn_amd import _lib, eeq as E
    gen = torch.Generator().manual_seed(n)
    side = 2.5 * n ** (1.0 / 3.0) + (30.0 if kind == "wide" else 6.0)
    cell = torch.tensor([[side, 0, 0], [0.2 * side, side, 0], [-0.1 * side, 0.15 * side, 1.1 * side]],
                        dtype=torch.float64)
    pos = (torch.rand(n, 3, dtype=torch.float64, generator=gen) @ cell * 1.4 - 3.0).to(DEV)
    rad = (0.5 + torch.rand(n, dtype=torch.float64, generator=gen)).to(DEV)
    u, w = (torch.randn(n, dtype=torch.float64, generator=gen).to(DEV) for _ in range(2))
    host = None if kind == "molecule" else E._host_cell(cell)
    alpha, cut = (0.0, 1e6) if host is None else (E.ewald_alpha(20.0), 20.0)
    stream = _lib.stream(pos.device)
    ref, rows = torch.empty_like(pos), torch.empty(n, 9, dtype=torch.float64, device=DEV)
    want = host is not None and kind != "no_cell_gradient"
    ins = (_lib.ptr(pos), n, host, _lib.ptr(rad), alpha, cut, _lib.ptr(u), _lib.ptr(w))
    _lib.call("xnn_eeq_real_grad", *ins, _lib.ptr(ref), _lib.ptr(rows) if host is not None else None, stream)
    need = ctypes.c_size_t(0)
    _lib.call("xnn_eeq_real_grad_pairs_work_size", n, ctypes.byref(need))
    outs = []
    for _ in range(2):
        work = torch.empty(need.value, dtype=torch.uint8, device=DEV)
        g, c = torch.empty_like(pos), torch.empty(9, dtype=torch.float64, device=DEV)
        _lib.call("xnn_eeq_real_grad_pairs", *ins, _lib.ptr(g), _lib.ptr(c) if want else None,
                  _lib.ptr(work), need.value, stream)
        outs.append((g, c))
    assert torch.equal(outs[0][0], outs[1][0])
    # terms of up to |K'| r^2 ~ 1 per pair with |u w| up to 16, a few roundings each
    tol = 1e-14 * 16 * max(n, 8)
    torch.testing.assert_close(outs[0][0], ref, rtol=0, atol=tol)
    if want:
        assert torch.equal(outs[0][1], outs[1][1])
        torch.testing.assert_close(outs[0][1], rows.sum(0), rtol=0, atol=tol * n)


def test_without_room_for_the_pairs_the_directed_kernel_runs(monkeypatch):
    from xnn_amd import _lib, eeq as E
    gen = torch.Generator().manual_seed(1)
    cell = 12.0 * torch.eye(3, dtype=torch.float64)
    pos = (torch.rand(100, 3, dtype=torch.float64, generator=gen) * 12.0).to(DEV)
    rad, u, v = (torch.rand(100, dtype=torch.float64, generator=gen).to(DEV) for _ in range(3))

    def grads():
        leaves = [pos.clone().requires_grad_(True), cell.to(DEV).requires_grad_(True)]
        out = E.real_apply_op(leaves[0], leaves[1], rad, v, None, E.ewald_alpha(20.0), 20.0)
        return torch.autograd.grad([out], leaves, [u])

    want = grads()
    need, empty = ctypes.c_size_t(0), torch.empty
    _lib.call("xnn_eeq_real_grad_pairs_work_size", 100, ctypes.byref(need))

    def full(*args, **kw):
        if args[0] == need.value:
            raise torch.cuda.OutOfMemoryError("no room")
        return empty(*args, **kw)

    before = _lib.calls.get("xnn_eeq_real_grad", 0)
    monkeypatch.setattr(torch, "empty", full)
    got = grads()
    monkeypatch.undo()
    assert _lib.calls.get("xnn_eeq_real_grad", 0) == before + 1
    # as above: terms of order one, a hundred of them an atom
    for a, b in zip(got, want):
        torch.testing.assert_close(a, b, rtol=0, atol=1e-14 * 16 * 100 * 100)
