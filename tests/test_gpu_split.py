"""The hop of few sites (one wave per direction) against the gathering kernel,
which a launch shape set by hand selects: the same bits for every opcode,
precision, link format and boundary, for odd counts of right-hand sides, whole
and partial workgroups, fields aligned to one value only, and whole CG solves
(their inner products come from the same kernel)."""
import pytest

from oracle import gauge as G
from oracle import rng as R

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

import gpt_amd as g  # noqa: E402
from gpt_amd import _lib, core  # noqa: E402

CASES = {
    "anti": dict(mass=0.1, csw_r=0.8, csw_t=0.8, boundary_phases=[1, 1, 1, -1]),
    "twist": dict(mass=0.1, csw_r=0.7, csw_t=0.9, xi_0=1.3, nu=0.9, isAnisotropic=True,
                  boundary_phases=[1j, -1, 0.6 + 0.8j, -1]),
    "open": dict(mass=0.2, csw_r=0.5, csw_t=0.5, cF=1.3, boundary_phases=[1, 1, 1, 0]),
    "plain": dict(mass=0.3, boundary_phases=[1, 1, 1, -1]),
}


def outputs(w, N, dtype, shift, vals):
    n = w.F_grid.Vh * 12 * N
    lib, h, s = _lib.load(), w.handle, core.stream_ptr()

    def field(m, fill=False):
        x = torch.zeros(2 * (m + shift), dtype=dtype, device=core.device())[2 * shift:]
        if fill:
            x.copy_(vals[:2 * m])
        return x

    out = []
    for opcode, cb, parts in [(2003, 0, 1), (2003, 1, 1), (2004, 0, 1), (2001, -1, 2), (2002, -1, 2), (4001, -1, 2)]:
        src, dst = field(parts * n, True), field(parts * n)
        _lib.check(lib.wc_apply_block(h, opcode, N, dst.data_ptr(), src.data_ptr(), cb, s))
        out.append(dst)
    for parity in (0, 1):
        for which in (0, 1, 2):
            src, dst = field(n, True), field(n)
            _lib.check(lib.wc_apply_mpc_block(h, parity, which, N, dst.data_ptr(), src.data_ptr(), s))
            out.append(dst)
    return out


@pytest.mark.parametrize("case", list(CASES))
@pytest.mark.parametrize("fd", [[4, 4, 4, 4], [2, 4, 16, 4], [12, 8, 8, 8]], ids=str)
def test_same_bits_as_the_gathering_kernel(fd, case):
    U = G.random_links(R.grid(fd), R.random("split"), scale=0.5)
    for prec in (g.double, g.single):
        for N, compress in ((1, False), (1, True), (3, False), (5, True)):
            w = g.qcd.fermion.wilson_clover(U, CASES[case], precision=prec, n_rhs=N, compress_links=compress)
            gen = torch.Generator(device="cuda").manual_seed(N)
            vals = torch.randn(4 * w.F_grid.Vh * 12 * N, generator=gen, device="cuda", dtype=prec.real_dtype)
            w.set_hop_shape((1, 1, 0, 1, 0))
            ref = outputs(w, N, prec.real_dtype, 0, vals)
            w.set_hop_shape(None)
            assert all(float(x.abs().sum()) > 0 for x in ref)
            for shift in (0, 1):
                for i, (a, b) in enumerate(zip(outputs(w, N, prec.real_dtype, shift, vals), ref)):
                    assert torch.equal(a, b), (fd, case, prec.__name__, N, shift, i)
            w.release()


@pytest.mark.parametrize("prec,eps", [(g.double, 1e-10), (g.single, 1e-5)], ids=["double", "single"])
@pytest.mark.parametrize("N", [1, 2])
def test_a_solve_and_its_graphs(prec, eps, N):
    fd = [4, 8, 6, 8]
    U = G.random_links(R.grid(fd), R.random("split_cg"), scale=0.5)
    w = g.qcd.fermion.wilson_clover(U, CASES["anti"], precision=prec, n_rhs=N)
    inv, pc = g.algorithms.inverter, g.qcd.fermion.preconditioner
    src = g.lattice(w.F_grid)
    src.data.normal_(generator=torch.Generator(device="cuda").manual_seed(5))
    got = []
    for shape, chunk in (((1, 1, 0, 1, 0), 1), (None, 1), (None, 0), (None, 0)):
        w.set_hop_shape(shape)
        w.set_iteration_chunk(chunk)
        cg = inv.cg(eps=eps, maxiter=500)
        x = g.eval(w.propagator(inv.preconditioned(pc.eo2_ne(), cg)) * src)
        assert cg.converged
        got.append((x.data.clone(), cg.history, cg.iterations))
    for x, hist, it in got[1:]:
        assert torch.equal(x, got[0][0]) and hist == got[0][1] and it == got[0][2]
