"""The three forms of the hop, set by name: which one a launch takes, and the same
bits from all of them for every opcode, epilogue (a solve's inner product among
them), precision, link format and boundary, on lattices of two sites a direction,
slices that are no whole number of 64-site blocks, waves that walk through one
slice or several, counts at the ends of each range and fields aligned to one value
only."""
import pytest

from oracle import gauge as G
from oracle import rng as R

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

import gpt_amd as g  # noqa: E402
from gpt_amd import _lib, core  # noqa: E402

inv = g.algorithms.inverter
pc = g.qcd.fermion.preconditioner

CASES = {
    "anti": dict(mass=0.1, csw_r=0.8, csw_t=0.8, boundary_phases=[1, 1, 1, -1]),
    "twist": dict(mass=0.1, csw_r=0.7, csw_t=0.9, xi_0=1.3, nu=0.9, isAnisotropic=True,
                  boundary_phases=[1j, -1, 0.6 + 0.8j, -1]),
    "open": dict(mass=0.2, csw_r=0.5, csw_t=0.5, cF=1.3, boundary_phases=[1, 1, 1, 0]),
    "plain": dict(mass=0.3, boundary_phases=[1, 1, 1, -1]),
}


def outputs(w, N, shift, vals):
    n = w.F_grid.Vh * 12 * N
    lib, h, s = _lib.load(), w.handle, core.stream_ptr()

    def field(m, fill=False):
        x = torch.zeros(2 * (m + shift), dtype=vals.dtype, device=core.device())[2 * shift:]
        if fill:
            x.copy_(vals[:2 * m])
        return x

    out = []
    for opcode, cb, parts in [(2003, 0, 1), (2003, 1, 1), (2004, 0, 1), (2004, 1, 1), (2001, -1, 2), (2002, -1, 2),
                              (3001, -1, 2), (4001, -1, 2)]:
        src, dst = field(parts * n, True), field(parts * n)
        _lib.check(lib.wc_apply_block(h, opcode, N, dst.data_ptr(), src.data_ptr(), cb, s))
        out.append(dst)
    for parity in (0, 1):
        for which in (0, 1, 2):
            src, dst = field(n, True), field(n)
            _lib.check(lib.wc_apply_mpc_block(h, parity, which, N, dst.data_ptr(), src.data_ptr(), s))
            out.append(dst)
    return out


def compare(form, fd, case, prec, N, compress):
    """the form's outputs and the gathering kernel's"""
    U = G.random_links(R.grid(fd), R.random("forms"), scale=0.5)
    w = g.qcd.fermion.wilson_clover(U, CASES[case], precision=prec, n_rhs=N, compress_links=compress)
    gen = torch.Generator(device="cuda").manual_seed(N)
    vals = torch.randn(4 * w.F_grid.Vh * 12 * N, generator=gen, device="cuda", dtype=prec.real_dtype)
    w.set_hop_form("gather")
    assert w.hop_form() == "gather"
    ref = outputs(w, N, 0, vals)
    w.set_hop_form(form)
    assert w.hop_form() == form
    for shift in (0, 1):
        for i, (a, b) in enumerate(zip(outputs(w, N, shift, vals), ref)):
            assert torch.equal(a, b), (fd, case, prec.__name__, N, compress, shift, i)
    if case != "open" or fd[3] > 2:  # two open slices leave no site
        assert all(float(x.abs().sum()) > 0 for x in ref)
    w.release()


@pytest.mark.parametrize("case", list(CASES))
@pytest.mark.parametrize("fd", [[4, 4, 4, 8], [2, 4, 16, 2], [6, 10, 2, 16], [12, 6, 4, 16]], ids=str)
def test_march(fd, case):
    for prec, counts in ((g.double, (8, 10, 12, 33, 64)), (g.single, (7, 8, 12, 13, 33, 64))):
        for N in counts:
            for compress in (False, True):
                compare("march", fd, case, prec, N, compress)


@pytest.mark.parametrize("fd,prec,N", [([16, 16, 16, 8], g.double, 12), ([16, 16, 16, 16], g.double, 10),
                                       ([16, 16, 16, 16], g.single, 13), ([16, 16, 16, 16], g.single, 8),
                                       ([20, 18, 6, 24], g.single, 12)], ids=str)
def test_march_through_several_slices(fd, prec, N):
    for case, compress in (("twist", False), ("anti", True)):
        compare("march", fd, case, prec, N, compress)


@pytest.mark.parametrize("case", list(CASES))
@pytest.mark.parametrize("fd", [[4, 4, 4, 4], [2, 4, 16, 2], [12, 8, 8, 8]], ids=str)
def test_split(fd, case):
    for prec in (g.double, g.single):
        for N in (1, 3, 5):
            for compress in (False, True):
                compare("split", fd, case, prec, N, compress)


@pytest.mark.parametrize("prec,N", [(g.double, 8), (g.double, 12), (g.single, 7), (g.single, 12)], ids=str)
@pytest.mark.parametrize("compress", [False, True])
def test_solves_and_their_graphs(prec, N, compress):
    """CG, with the inner products of the hop's epilogue: the same histories and
    solutions; a form set between two solves is not replayed from an old graph"""
    fd = [8, 4, 6, 8]
    U = G.random_links(R.grid(fd), R.random("forms_cg"), scale=0.5)
    w = g.qcd.fermion.wilson_clover(U, CASES["anti"], precision=prec, n_rhs=N, compress_links=compress)
    src = g.lattice(w.F_grid)
    src.data.normal_(generator=torch.Generator(device="cuda").manual_seed(5))
    got = []
    for form, chunk in (("gather", 1), ("march", 1), ("march", 0), ("split", 0), ("gather", 0), ("march", 0)):
        w.set_hop_form(form)
        w.set_iteration_chunk(chunk)
        assert w.hop_form() == form
        cg = inv.cg(eps=1e-9 if prec is g.double else 1e-5, maxiter=500)
        x = g.eval(w.propagator(inv.preconditioned(pc.eo2_ne(), cg)) * src)
        assert cg.converged
        got.append((x.data.clone(), cg.history, cg.iterations))
    for x, hist, it in got[1:]:
        assert torch.equal(x, got[0][0]) and hist == got[0][1] and it == got[0][2]


def test_mixed_solve_on_each_form():
    """the FP32 inner operator of a mixed solve, 12 right-hand sides"""
    fd = [8, 8, 8, 8]
    U = G.smooth_links(fd, 0.3, 9001)
    w = g.qcd.fermion.wilson_clover(U, CASES["anti"], n_rhs=12)
    src = g.lattice(w.F_grid)
    src.data.normal_(generator=torch.Generator(device="cuda").manual_seed(6))
    got = []
    for form in ("gather", "march", "split"):
        m = inv.cg_mixed(eps=1e-10, maxiter=2000)
        for x in (w, m.inner_operator(w)):
            x.set_hop_form(form, n_rhs=12)
        assert m.inner_operator(w).hop_form(12) == form
        x = g.eval(w.propagator(inv.preconditioned(pc.eo2_ne(), m)) * src)
        assert m.converged
        got.append((x.data.clone(), m.iterations, m.reliable_updates))
    for x, it, up in got[1:]:
        assert torch.equal(x, got[0][0]) and it == got[0][1] and up == got[0][2]


def test_which_form_a_hop_takes():
    small = G.random_links(R.grid([8, 8, 8, 8]), R.random("forms"), scale=0.5)
    for prec, most in ((g.double, 8), (g.single, 16)):  # pairs 2048 N
        w = g.qcd.fermion.wilson_clover(small, CASES["anti"], precision=prec)
        assert w.hop_form(most) == "split" and w.hop_form(most + 1) != "split"
        w.set_hop_form("split", n_rhs=most + 1)
        assert w.hop_form(most + 1) == "gather"  # it has no such form
        w.set_hop_form("march", n_rhs=1)
        assert w.hop_form(1) == "gather"
        w.release()
    # a shape is the gathering kernel's, also the one in use; a form holds beside it
    w = g.qcd.fermion.wilson_clover(small, CASES["anti"])
    shape = w.hop_shape()
    assert w.hop_form() == "split"
    w.set_hop_shape(shape)
    assert w.hop_form() == "gather" and w.hop_shape() == shape
    w.set_hop_form("auto")
    assert w.hop_form() == "split" and w.hop_shape() == shape
    w.set_hop_shape((1, 2, 4, 1, 0))
    assert w.hop_form() == "split" and w.hop_shape() == (1, 2, 4, 1, 0)
    w.set_hop_form(None)
    assert w.hop_form() == "gather"
    w.set_hop_shape(None)
    assert w.hop_form() == "split" and w.hop_shape() == shape
    w.release()
    large = g.qcd.fermion.wilson_clover(G.smooth_links([16, 16, 16, 16], 0.3, 9002), CASES["anti"], n_rhs=12)
    assert large.hop_form() == "march" and large.hop_form(9) == "gather" and large.hop_form(1) == "gather"
    large.set_hop_shape(large.hop_shape())
    assert large.hop_form() == "gather"
    large.set_hop_form("auto")
    assert large.hop_form() == "march"
    with pytest.raises(RuntimeError, match="form"):
        _lib.check(_lib.load().wc_set_hop_form(large.handle, 1, 5))
    with pytest.raises(RuntimeError, match="nrhs"):
        _lib.check(_lib.load().wc_set_hop_form(large.handle, 0, 1))
    with pytest.raises(ValueError):
        large.set_hop_form("other")
