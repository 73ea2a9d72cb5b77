"""unpack into any container that gives its fields by number, not lists alone."""
import collections

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

import gpt_amd as g  # noqa: E402
from gpt_amd.qcd.fermion.operator import pack, unpack  # noqa: E402


class by_number:
    def __init__(self, fields):
        self.fields = fields

    def __getitem__(self, r):
        return self.fields[r]


@pytest.mark.parametrize("kind", [list, tuple, collections.deque, lambda f: dict(enumerate(f)), by_number],
                         ids=["list", "tuple", "deque", "dict", "by_number"])
def test_containers(kind):
    grid = g.grid([4, 4, 4, 6], g.double)
    src = [g.lattice(grid) for _ in range(3)]
    for i, f in enumerate(src):
        f.data.normal_(generator=torch.Generator(device="cuda").manual_seed(i))
    P = pack(src)
    dst = kind([g.lattice(grid) for _ in range(4)])  # one more than needed
    dst[3].data.zero_()
    assert unpack(P, dst) is dst
    assert all(torch.equal(dst[r].data, src[r].data) for r in range(3)) and float(dst[3].data.abs().max()) == 0
