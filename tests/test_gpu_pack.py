"""Lists of fields to many-RHS fields and back: the same values as one strided
copy per field, for every count and precision, full and half fields, and the
forms that a kernel cannot take (views, another precision, a field given twice)."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

import gpt_amd as g  # noqa: E402
from gpt_amd.core import lattice  # noqa: E402
from gpt_amd.qcd.fermion.operator import pack, unpack  # noqa: E402


def random_fields(grid, n, cb=None):
    out = []
    for r in range(n):
        x = lattice(grid)
        if cb is not None:
            x.checkerboard(cb)
        x.data.normal_(generator=torch.Generator(device="cuda").manual_seed(r + 1))
        out.append(x)
    return out


def copies(fields):
    return torch.cat([f.data for f in fields], dim=-2)


@pytest.mark.parametrize("prec", [g.double, g.single], ids=["double", "single"])
@pytest.mark.parametrize("half", [False, True], ids=["full", "half"])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 7, 8, 12, 31, 32, 33, 45, 64])
def test_there_and_back(n, half, prec):
    grid = g.grid([4, 4, 12, 6], prec)
    cb = None
    if half:
        grid, cb = grid.checkerboarded(g.redblack), g.odd
    fields = random_fields(grid, n, cb)
    P = pack(fields)
    assert P.grid.nrhs == n and P.checkerboard() is fields[0].checkerboard()
    assert torch.equal(P.data, copies(fields))
    back = unpack(P)
    given = random_fields(grid, n + 1, g.even if half else None)
    last = given[n].data.clone()
    assert unpack(P, given) is given and torch.equal(given[n].data, last)
    for r in range(n):
        for x in (back[r], given[r]):
            assert torch.equal(x.data, fields[r].data) and x.checkerboard() is fields[r].checkerboard()


def test_values_at_an_odd_address():
    grid = g.grid([4, 4, 4, 4], g.double)
    fields = random_fields(grid, 5)
    moved = random_fields(grid, 5)
    for m, f in zip(moved, fields):
        m.data = torch.empty(f.data.numel() + 1, dtype=f.data.dtype, device="cuda")[1:].view(f.data.shape)
        m.data.copy_(f.data)
    P = pack(moved)
    assert torch.equal(P.data, copies(fields))
    for m in moved:
        m.data.zero_()
    unpack(P, moved)
    assert all(torch.equal(m.data, f.data) for m, f in zip(moved, fields))


def test_general_forms():
    grid, gs = g.grid([4, 4, 4, 4], g.double), g.grid([4, 4, 4, 4], g.single)
    a, b, c = random_fields(grid, 3)
    assert torch.equal(pack([a, b, a]).data, copies([a, b, a]))
    v = lattice(grid)
    v.data = torch.stack([b.data, c.data], -1)[..., 1]  # strided
    assert torch.equal(pack([a, v]).data, copies([a, c]))
    s, = random_fields(gs, 1)
    assert torch.equal(pack([a, s]).data, torch.cat([a.data, s.data.double()], -2))
    P = pack([a, b, c])
    x, y = lattice(grid), lattice(grid)
    unpack(P, [x, y, x])  # the last one wins
    assert torch.equal(x.data, c.data) and torch.equal(y.data, b.data)
    lo = [lattice(gs) for _ in range(3)]
    unpack(P, lo)
    assert torch.equal(lo[1].data, b.data.float())
    with pytest.raises(ValueError):
        pack([a, lattice(g.grid([4, 4, 4, 8], g.double))])
    with pytest.raises(IndexError):
        unpack(P, [x, y])
