"""g.trace and g.slice of values that lie in host memory, on a machine without a
GPU too, and directions given as other numbers than int: against numpy."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import gpt_amd as g  # noqa: E402
from gpt_amd import core  # noqa: E402

GRID = g.grid([4, 6, 8, 4], g.double)


def host_field(seed, prec=g.double):
    p = core.mspincolor_lattice.__new__(core.mspincolor_lattice)
    p.grid = g.grid(GRID.fdimensions, prec)
    rng = np.random.default_rng(seed)
    a = rng.standard_normal((GRID.gsites, 4, 4, 3, 3)) + 1j * rng.standard_normal((GRID.gsites, 4, 4, 3, 3))
    p.data = torch.from_numpy(a.astype(prec.complex_dtype))
    return p


@pytest.mark.parametrize("prec", [g.double, g.single], ids=["double", "single"])
def test_values_in_host_memory(prec):
    a, b = host_field(1, prec), host_field(2, prec)
    x, y = (p.data.numpy().astype(np.complex128).reshape(GRID.gsites, -1) for p in (a, b))
    want = (x * y.conj()).sum(1)
    # 144 products and sums of numbers of order 1
    assert np.abs(g.trace(a * g.adj(b)).data.numpy() - want).max() <= 148 * 2.3e-16 * 40
    tr = core.site_scalar(GRID, torch.from_numpy(want))
    f = want.reshape(GRID.fdimensions[::-1])
    for dim in range(4):
        other = tuple(d for d in range(4) if d != 3 - dim)
        ref = f.sum(other)
        assert np.abs(np.array(g.slice(tr, dim)) - ref).max() <= f.size * 2.3e-16 * np.abs(f).max()


@pytest.mark.parametrize("kind", [float, np.float64, np.int64, np.uint8, torch.tensor], ids=lambda k: k.__name__)
def test_directions_as_other_numbers(kind):
    rng = np.random.default_rng(3)
    tr = core.site_scalar(GRID, torch.from_numpy(rng.standard_normal(GRID.gsites) + 0j))
    for dim in range(4):
        assert g.slice(tr, kind(dim)) == g.slice(tr, dim)
    for dim in (4, -1):
        with pytest.raises(TypeError):
            g.slice(tr, kind(dim) if kind is not np.uint8 else 4)


@pytest.mark.parametrize("fd,dims", [([4, 4, 4, 4], range(4)), ([8, 8, 8, 16], range(4)),
                                     ([32, 32, 16, 14], range(4)), ([32, 32, 16, 16], (0, 3))], ids=str)
def test_general_sums_look_at_nothing_else(fd, dims, monkeypatch):
    """where the general sum is as fast as the kernel, below 2^18 sites and along t"""
    def fail(*_):
        raise AssertionError("a small field was checked for the kernel")

    monkeypatch.setattr(core, "direct", fail)
    grid = g.grid(fd, g.double)
    tr = core.site_scalar(grid, torch.ones(grid.gsites, dtype=torch.complex128))
    for dim in dims:
        assert g.slice(tr, dim) == [grid.gsites / fd[dim]] * fd[dim]
