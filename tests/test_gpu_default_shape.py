"""The launch shapes that hops have before any tuning, against one wave per
workgroup and one right-hand side per thread: the same bits on lattices around
the sizes where the shape changes, for every count class, both link formats and
FP16 and bfloat16 spinors."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

import gpt_amd as g  # noqa: E402
from gpt_amd import _lib, core  # noqa: E402

P = dict(mass=0.1, csw_r=0.9, csw_t=0.9, boundary_phases=[1, 1, 1, -1])


def operator(fd, prec, n, compress):
    grid = g.grid(fd, g.double)
    gen = torch.Generator(device="cuda").manual_seed(7)
    U = []
    for _ in range(4):
        q = torch.randn(grid.gsites, 3, 3, dtype=torch.complex128, device="cuda", generator=gen)
        a = q[:, 0] / q[:, 0].norm(dim=-1, keepdim=True)
        b = q[:, 1] - (a.conj() * q[:, 1]).sum(-1, keepdim=True) * a
        b = b / b.norm(dim=-1, keepdim=True)
        U.append(g.qcd.gauge.link_field(grid, torch.stack([a, b, torch.linalg.cross(a, b).conj()], 1)))
    return g.qcd.fermion.wilson_clover(U, P, precision=prec, n_rhs=n, compress_links=compress)


def run(w, n, storage):
    lib, s = _lib.load(), core.stream_ptr()
    m = w.F_grid.Vh * 12 * n
    dt = w.F_grid.precision.real_dtype
    x = torch.randn(4 * m, dtype=dt, device="cuda", generator=torch.Generator(device="cuda").manual_seed(n))
    y = torch.zeros(2 * m, dtype=dt, device="cuda")
    if storage is None:
        z = torch.zeros(4 * m, dtype=dt, device="cuda")
        _lib.check(lib.wc_apply_mpc_block(w.handle, 0, 2, n, y.data_ptr(), x.data_ptr(), s))
        _lib.check(lib.wc_apply_block(w.handle, 2002, n, z.data_ptr(), x.data_ptr(), -1, s))
        return y, z
    half = x[:2 * m].to({"half": torch.float16, "bf16": torch.bfloat16}[storage]).reshape(-1, 12, 64, n, 2)
    return (w.mpc_ne_s16(half, 0, storage, n),)


SIZES = [[8, 8, 8, 16], [16, 12, 16, 16], [10, 18, 16, 32], [16, 16, 24, 32], [32, 32, 32, 16]]


@pytest.mark.parametrize("fd", SIZES, ids=str)
@pytest.mark.parametrize("prec", ["double", "single", "half", "bf16"])
def test_same_bits_as_the_plainest_shape(fd, prec):
    storage = prec if prec in ("half", "bf16") else None
    big = fd == SIZES[-1]
    for n in (1, 2, 4) if big else (1, 2, 3, 4, 5, 6, 7, 8, 9, 13):
        for compress in (False, True):
            w = operator(fd, g.double if prec == "double" else g.single, n, compress)
            got = run(w, n, storage)
            w.set_hop_shape((1, 1, 0, 1, 0))
            for a, b in zip(got, run(w, n, storage)):
                assert float(a.abs().max()) > 0 and torch.equal(a, b), (n, compress)
            w.release()
