"""g.slice on lattices large enough for its kernel, in every direction, and the
kernel on all kinds of shapes, against numpy in extended precision."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

import gpt_amd as g  # noqa: E402
from gpt_amd import _lib, core  # noqa: E402

L = np.clongdouble


def values(n, seed):
    return torch.randn(n, generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda",
                       dtype=torch.complex128)


@pytest.mark.parametrize("fd", [[16, 18, 30, 32], [20, 32, 16, 26], [2, 64, 64, 34], [64, 64, 32, 2]], ids=str)
def test_slices(fd):
    grid = g.grid(fd, g.double)
    tr = core.site_scalar(grid, values(grid.gsites, 1))
    f = tr.data.cpu().numpy().astype(L).reshape(fd[::-1])
    for dim in range(4):
        other = tuple(d for d in range(4) if d != 3 - dim)
        # FP64 sums in any order
        assert np.all(np.abs(np.array(g.slice(tr, dim)) - f.sum(other)) <= f.size // fd[dim] * 2.3e-16
                      * np.abs(f).sum(other))


@pytest.mark.parametrize("outer,n,inner", [(1, 1, 1), (1, 3, 1), (7, 2, 5), (1, 66, 8), (64, 4, 64), (5, 130, 257),
                                           (1, 2, 40000), (3000, 3, 7)])
def test_kernel(outer, n, inner):
    x = values(outer * n * inner, 2)
    work = torch.empty((17, n), dtype=torch.complex128, device="cuda")
    _lib.check(_lib.load().wc_slice_sum(outer, n, inner, x.data_ptr(), work[1].data_ptr(), work.data_ptr(),
                                        core.stream_ptr()))
    f = x.cpu().numpy().astype(L).reshape(outer, n, inner)
    assert np.all(np.abs(work[0].cpu().numpy() - f.sum((0, 2))) <= outer * inner * 2.3e-16 * np.abs(f).sum((0, 2)))
