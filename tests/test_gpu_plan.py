"""The edge plan (``xnn_graph_plan``): both CSR orderings, the structures' layout and the
atom order against NumPy's stable sorts, at the edges of its row sorts and scans."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _lists(name, rng):
    """``(senders, receivers, atoms)`` of one case."""
    def random(n, e):
        return rng.integers(0, n, e), rng.integers(0, n, e), n

    if name == "empty":
        return np.zeros(0, int), np.zeros(0, int), 5
    if name == "one":
        return np.array([0]), np.array([0]), 1
    if name == "ungrouped":                      # rows of about 40, many waves a row's edge
        return random(3001, 120_007)
    if name == "grouped":
        s, d, n = random(3001, 120_007)
        return s, np.sort(d), n
    if name == "two_tiles":                      # more rows than one scan block takes
        return random(20_011, 33_333)
    if name == "rows_64_65":
        d = np.repeat(np.arange(4), [63, 64, 65, 128])
        return rng.permutation(d), rng.permutation(d), 4
    if name == "rows_1024_1025":                 # the last row of each sort
        d = np.repeat(np.arange(5), [1023, 1024, 1025, 0, 5000])
        return rng.permutation(d), d, 5
    if name == "sorted_hub":                     # long runs of one sender
        return np.sort(random(50, 60_000)[0]), random(50, 60_000)[1], 50
    assert name == "library"                     # mean rows above 8,192
    return random(3, 30_000)


@pytest.mark.parametrize("name", ["empty", "one", "ungrouped", "grouped", "two_tiles", "rows_64_65",
                                  "rows_1024_1025", "sorted_hub", "library"])
def test_plan_orderings_are_stable_sorts(name):
    from xnn_amd.plan import build_plan
    rng = np.random.default_rng(3)
    src, dst, n = _lists(name, rng)
    shift = rng.integers(-512, 512, (len(src), 3))
    pos = rng.uniform(-20, 20, (n, 3))
    cut = n // 3
    plan = build_plan(torch.tensor(np.stack([src, dst]), device=DEV), torch.tensor(shift, device=DEV), n,
                      torch.tensor(np.arange(n) >= cut, device=DEV).long(),
                      torch.tensor([cut, n - cut], device=DEV), torch.tensor(pos, device=DEV))
    assert np.array_equal(plan.src.cpu(), src) and np.array_equal(plan.dst.cpu(), dst)
    packed = plan.shift.cpu().numpy().astype(np.int64)
    for a in range(3):
        field = (packed >> (10 * a)) & 1023
        assert np.array_equal(np.where(field > 511, field - 1024, field), shift[:, a])
    for key, ptr, perm in ((src, plan.ptr_src, plan.perm_src), (dst, plan.ptr_dst, plan.perm_dst)):
        assert np.array_equal(ptr.cpu(), np.concatenate([[0], np.cumsum(np.bincount(key, minlength=n))]))
        order = np.argsort(key, kind="stable")
        got = np.arange(len(key)) if perm is None else perm.cpu().numpy()
        assert np.array_equal(got, order)
    assert (plan.perm_dst is None) == bool((np.diff(dst) >= 0).all())
    assert plan.node_ptr.tolist() == [0, cut, n]
    assert np.array_equal(plan.batch32.cpu(), np.arange(n) >= cut)
    visit = plan.visit.cpu().numpy()
    assert np.array_equal(np.sort(visit), np.arange(n))
    assert (np.diff((visit >= cut).astype(int)) >= 0).all()           # structure by structure


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_visit_order_follows_the_cell(dtype):
    """Atoms of one bin stay together for any lattice: the cubes of a 16^3 crystal of 8 atoms
    each are visited one whole cube after another, also from images outside the cell and with
    a position that is not finite."""
    from xnn_amd.plan import build_plan
    rng = np.random.default_rng(1)
    cell = np.array([[16.0, 0, 0], [3.0, 15.0, 0], [-2.0, 1.0, 17.0]])
    cube = rng.permutation(np.repeat(np.arange(16 ** 3), 8))
    frac = (np.stack([cube // 256, cube // 16 % 16, cube % 16], 1) + rng.uniform(.2, .8, (len(cube), 3))) / 16
    pos = (frac + rng.integers(-2, 3, frac.shape)) @ cell
    n = len(pos)
    none = torch.zeros((2, 0), dtype=torch.long, device=DEV)
    t = torch.tensor(pos, device=DEV, dtype=dtype)
    c = torch.tensor(cell, device=DEV, dtype=dtype)[None]
    visit = build_plan(none, None, n, pos=t, cell=c).visit.cpu().numpy()
    assert (cube[visit].reshape(-1, 8) == cube[visit].reshape(-1, 8)[:, :1]).all()
    t[5, 1] = float("nan")
    assert np.array_equal(np.sort(build_plan(none, None, n, pos=t, cell=c).visit.cpu().numpy()),
                          np.arange(n))


def test_a_batch_or_positions_that_miss_atoms_are_refused():
    """The plan's kernel reads one entry an atom; refused on the host, before any launch."""
    from xnn_amd.plan import build_plan
    none = torch.zeros((2, 0), dtype=torch.long, device=DEV)
    with pytest.raises(ValueError, match="batch holds 4"):
        build_plan(none, None, 5, torch.zeros(4, dtype=torch.long, device=DEV))
    for shape in ((4, 3), (5, 2), (6, 3)):
        with pytest.raises(ValueError, match="positions"):
            build_plan(none, None, 5, pos=torch.zeros(shape, device=DEV))
    plan = build_plan(none, None, 5, pos=torch.rand((5, 3)))           # from the host
    assert sorted(plan.visit.tolist()) == [0, 1, 2, 3, 4]


def test_edge_plan_reports_errors_only():
    """``xnn_edge_plan``'s flag is 0 for a list that is not grouped by receiver."""
    import ctypes
    from xnn_amd import _lib
    rng = np.random.default_rng(0)
    n, e = 300, 5000
    ei = torch.tensor(rng.integers(0, n, (2, e)), device=DEV)
    out = [torch.empty(k, dtype=torch.int32, device=DEV) for k in (e, e, e, n + 1, e, n + 1, e, 1)]
    need = int(_lib.load().xnn_edge_plan_workspace_bytes(e, n))
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    _lib.call("xnn_edge_plan", _lib.ptr(ei), None, e, n, *[_lib.ptr(t) for t in out], _lib.ptr(ws),
              ctypes.c_size_t(need), _lib.stream(torch.device(DEV)))
    assert out[7].item() == 0
    for row, ptr, perm in ((1, out[3], out[4]), (0, out[5], out[6])):
        key = ei[row].cpu().numpy()
        assert np.array_equal(ptr.cpu(), np.concatenate([[0], np.cumsum(np.bincount(key, minlength=n))]))
        assert np.array_equal(perm.cpu(), np.argsort(key, kind="stable"))


@pytest.mark.parametrize("e,hubs", [
    (200_000, [1024, 1025, 1500, 90_000]),            # one window of 253,952 ids
    (700_000, [1024, 1025, 5000, 2000, 300_000]),     # three, some of a row's empty
    (300_000, [299_990]),                             # nearly all
    (5_300_000, [1100, 10_751, 10_752, 12_000, 40_000]),  # 21: a wave sorts up to 10,751 ids
])
@pytest.mark.parametrize("scattered", [True, False])
def test_rows_of_any_length_are_sorted(e, hubs, scattered):
    """A few long rows among short ones, their ids all over the list or in one stretch."""
    from xnn_amd.plan import build_plan
    rng = np.random.default_rng(e + len(hubs))
    n = 5000
    key = rng.integers(len(hubs), n, e)
    at = rng.permutation(e) if scattered else np.roll(np.arange(e), e // 3)
    s0 = 0
    for row, length in enumerate(hubs):
        key[at[s0:s0 + length]] = row
        s0 += length
    other = rng.permutation(key)
    plan = build_plan(torch.tensor(np.stack([key, other]), device=DEV), None, n)
    for k, ptr, perm in ((key, plan.ptr_src, plan.perm_src), (other, plan.ptr_dst, plan.perm_dst)):
        assert np.array_equal(ptr.cpu(), np.concatenate([[0], np.cumsum(np.bincount(k, minlength=n))]))
        assert np.array_equal(perm.cpu(), np.argsort(k, kind="stable"))


def test_visit_order_of_one_crowded_bin():
    """Atoms in one corner of a wide cell share a bin: they are visited in their order."""
    from xnn_amd.plan import build_plan
    none = torch.zeros((2, 0), dtype=torch.long, device=DEV)
    pos = torch.rand((30_000, 3), device=DEV, dtype=torch.float64)
    cell = torch.eye(3, device=DEV, dtype=torch.float64)[None] * 1e4
    assert torch.equal(build_plan(none, None, 30_000, pos=pos, cell=cell).visit.cpu(),
                       torch.arange(30_000, dtype=torch.int32))


@pytest.mark.parametrize("n,e", [(1, 1), (64, 60), (65, 130), (1000, 3999), (1000, 4000), (40_000, 9000)])
def test_rows_of_few_ids(n, e):
    """A lane a row below four ids a row on the average; some rows are longer than its eight."""
    from xnn_amd.plan import build_plan
    rng = np.random.default_rng(n + e)
    key, other = rng.integers(0, n, e), rng.integers(0, n, e)
    key[rng.permutation(e)[:e // 3]] = n // 2
    other[rng.permutation(e)[:min(e, 9)]] = n - 1
    plan = build_plan(torch.tensor(np.stack([key, other]), device=DEV), None, n)
    for k, perm in ((key, plan.perm_src), (other, plan.perm_dst)):
        got = np.arange(e) if perm is None else perm.cpu()
        assert np.array_equal(got, np.argsort(k, kind="stable"))
