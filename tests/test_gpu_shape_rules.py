"""The launch shapes before any tuning, on both sides of each line of their rules."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

import gpt_amd as g  # noqa: E402

P = dict(mass=0.1, boundary_phases=[1, 1, 1, -1])


def shape(fd, prec, n, compress):
    grid = g.grid(fd, g.double)
    one = torch.eye(3, dtype=torch.complex128, device="cuda").expand(grid.gsites, 3, 3).contiguous()
    w = g.qcd.fermion.wilson_clover([g.qcd.gauge.link_field(grid, one) for _ in range(4)], P, precision=prec,
                                    n_rhs=n, compress_links=compress)
    out = w.hop_shape()
    w.release()
    return out


@pytest.mark.parametrize("fd,compress,want", [
    # in the cache: as many waves a workgroup as still fill the CUs evenly
    ([16, 16, 16, 16], False, (1, 2, 0, 1, 2)), ([10, 18, 16, 24], False, (1, 1, 0, 1, 0)),
    ([14, 16, 16, 24], False, (1, 1, 0, 1, 0)), ([16, 16, 16, 24], False, (1, 4, 0, 1, 2)),
    ([16, 16, 16, 32], True, (1, 4, 0, 1, 2)), ([12, 16, 20, 40], False, (1, 2, 0, 1, 2)),
    ([20, 20, 16, 32], False, (1, 4, 0, 1, 2)), ([16, 24, 32, 32], True, (1, 4, 0, 1, 2)),
    # slices that outgrow the L2, or beyond the cache
    ([24, 24, 24, 24], False, (1, 1, 4, 1, 2)), ([24, 24, 24, 24], True, (1, 1, 4, 1, 2)),
    ([16, 24, 32, 32], False, (1, 1, 4, 1, 2)), ([24, 24, 24, 48], True, (1, 1, 4, 1, 2)),
    ([24, 24, 32, 64], False, (1, 1, 4, 1, 0)), ([24, 24, 32, 64], True, (1, 1, 4, 1, 0)),
    ([32, 32, 32, 32], False, (1, 1, 4, 1, 2)), ([32, 32, 64, 32], False, (1, 1, 4, 1, 0)),
], ids=str)
def test_double_one(fd, compress, want):
    assert shape(fd, g.double, 1, compress) == want


@pytest.mark.parametrize("fd,compress,want", [
    ([12, 12, 12, 24], False, (1, 1, 4, 1, 0)), ([16, 16, 16, 16], False, (1, 4, 4, 1, 0)),
    ([10, 18, 16, 24], False, (1, 2, 4, 1, 0)), ([12, 16, 16, 24], False, (1, 2, 4, 1, 0)),
    ([14, 16, 16, 24], False, (1, 2, 4, 1, 0)), ([16, 16, 16, 32], False, (1, 8, 4, 1, 0)),
    ([12, 16, 20, 40], False, (1, 4, 4, 1, 0)), ([16, 16, 16, 48], False, (1, 4, 4, 1, 0)),
    ([10, 18, 16, 32], False, (1, 2, 4, 1, 0)), ([16, 16, 16, 24], False, (1, 4, 4, 1, 0)),
    ([20, 20, 16, 32], False, (1, 8, 4, 1, 0)),
    ([24, 24, 24, 24], True, (1, 1, 4, 1, 0)), ([24, 24, 24, 24], False, (1, 1, 4, 1, 0)),
    ([28, 28, 28, 32], False, (1, 1, 4, 1, 0)), ([32, 32, 32, 32], True, (1, 2, 4, 1, 0)),
    ([16, 32, 32, 32], False, (1, 1, 4, 1, 0)), ([64, 32, 32, 16], False, (1, 4, 4, 1, 0)),
], ids=str)
def test_double_two(fd, compress, want):
    assert shape(fd, g.double, 2, compress) == want


@pytest.mark.parametrize("fd,compress,want", [
    ([12, 12, 12, 24], False, (1, 2, 4, 1, 0)), ([16, 16, 16, 20], False, (1, 2, 4, 1, 0)),
    ([14, 16, 16, 24], False, (1, 4, 4, 1, 0)), ([10, 18, 16, 32], True, (1, 4, 4, 1, 0)),
    ([16, 16, 16, 32], True, (1, 2, 4, 1, 0)), ([18, 18, 16, 24], False, (1, 4, 4, 1, 0)),
    ([24, 24, 24, 24], True, (1, 4, 4, 1, 0)),
], ids=str)
def test_double_four(fd, compress, want):
    assert shape(fd, g.double, 4, compress) == want


@pytest.mark.parametrize("fd,compress,want", [
    ([8, 16, 16, 32], False, (2, 4, 0, 1, 0)), ([10, 18, 16, 24], True, (2, 1, 0, 1, 0)),
    ([12, 16, 16, 24], True, (2, 2, 0, 1, 0)), ([10, 20, 16, 32], False, (2, 4, 0, 1, 0)),
    ([24, 24, 24, 48], False, (2, 2, 0, 1, 0)), ([32, 32, 32, 32], False, (2, 2, 0, 1, 0)),
    ([20, 32, 32, 32], False, (2, 4, 0, 1, 0)), ([28, 28, 28, 56], True, (2, 4, 0, 1, 0)),
], ids=str)
def test_single_three(fd, compress, want):
    assert shape(fd, g.single, 3, compress) == want
