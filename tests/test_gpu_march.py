"""The t-marching hop (many right-hand sides) against the gathering kernel,
which a launch shape set by hand selects: the same bits, for every epilogue,
both link formats, open, twisted and antiperiodic boundaries, lattices of two
sites a direction, slices that are no whole number of 64-site blocks, counts at
the ends of its range and fields aligned to one value only."""
import pytest

from oracle import gauge as G
from oracle import rng as R

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

import gpt_amd as g  # noqa: E402
from gpt_amd import _lib, core  # noqa: E402

ANTI = dict(mass=0.1, csw_r=0.8, csw_t=0.8, boundary_phases=[1, 1, 1, -1])
TWIST = dict(mass=0.1, csw_r=0.7, csw_t=0.9, xi_0=1.3, nu=0.9, isAnisotropic=True,
             boundary_phases=[1j, -1, 0.6 + 0.8j, -1])
OPEN = dict(mass=0.2, csw_r=0.5, csw_t=0.5, cF=1.3, boundary_phases=[1, 1, 1, 0])
PLAIN = dict(mass=0.3, boundary_phases=[1, 1, 1, -1])


def values(n, dtype, shift, fill=None):
    flat = torch.zeros(2 * (n + shift), dtype=dtype, device=core.device())
    x = flat[2 * shift:]
    if fill is not None:
        x.copy_(fill)
    return x


def outputs(w, N, dtype, shift, vals):
    n = w.F_grid.Vh * 12 * N
    lib, h, s = _lib.load(), w.handle, core.stream_ptr()
    out = []
    for opcode, cb, parts in [(2003, 0, 1), (2003, 1, 1), (2004, 1, 1), (2001, -1, 2), (2002, -1, 2), (3001, -1, 2)]:
        src, dst = values(parts * n, dtype, shift, vals[:2 * parts * n]), values(parts * n, dtype, shift)
        _lib.check(lib.wc_apply_block(h, opcode, N, dst.data_ptr(), src.data_ptr(), cb, s))
        out.append(dst)
    for parity in (0, 1):
        for which in (0, 1, 2):
            src, dst = values(n, dtype, shift, vals[:2 * n]), values(n, dtype, shift)
            _lib.check(lib.wc_apply_mpc_block(h, parity, which, N, dst.data_ptr(), src.data_ptr(), s))
            out.append(dst)
    return out


@pytest.mark.parametrize("params", [ANTI, TWIST, OPEN, PLAIN], ids=["anti", "twist", "open", "plain"])
@pytest.mark.parametrize("fd", [[4, 4, 4, 8], [2, 4, 16, 2], [6, 10, 2, 16], [12, 6, 4, 16]], ids=str)
def test_same_bits_as_the_gathering_kernel(fd, params):
    U = G.random_links(R.grid(fd), R.random("march"), scale=0.5)
    for prec, counts in ((g.double, (8, 10, 12, 33, 64)), (g.single, (7, 8, 12, 13, 64))):
        for N in counts:
            w = g.qcd.fermion.wilson_clover(U, params, precision=prec, n_rhs=N, compress_links=N in (12, 33, 13))
            gen = torch.Generator(device="cuda").manual_seed(N)
            vals = torch.randn(4 * w.F_grid.Vh * 12 * N, generator=gen, device="cuda", dtype=prec.real_dtype)
            w.set_hop_shape((1, 1, 4, 1, 0))
            ref = outputs(w, N, prec.real_dtype, 0, vals)
            w.set_hop_shape(None)
            for shift in (0, 1):
                for i, (a, b) in enumerate(zip(outputs(w, N, prec.real_dtype, shift, vals), ref)):
                    assert torch.equal(a, b), (fd, prec.__name__, N, shift, i)
            if params is not OPEN or fd[3] > 2:  # two open slices leave no site
                assert all(float(x.abs().sum()) > 0 for x in ref)
            w.release()


@pytest.mark.parametrize("prec,N", [(g.double, 12), (g.single, 13)], ids=["double", "single"])
def test_several_slices_a_wave(prec, N):
    """slices large enough that a wave walks through several of them"""
    fd = [16, 16, 16, 8]
    U = G.random_links(R.grid(fd), R.random("march_walk"), scale=0.5)
    w = g.qcd.fermion.wilson_clover(U, TWIST, precision=prec, n_rhs=N)
    gen = torch.Generator(device="cuda").manual_seed(N)
    vals = torch.randn(4 * w.F_grid.Vh * 12 * N, generator=gen, device="cuda", dtype=prec.real_dtype)
    w.set_hop_shape((1, 1, 4, 1, 0))
    ref = outputs(w, N, prec.real_dtype, 0, vals)
    w.set_hop_shape(None)
    for i, (a, b) in enumerate(zip(outputs(w, N, prec.real_dtype, 0, vals), ref)):
        assert torch.equal(a, b), i


@pytest.mark.parametrize("N", [9, 12])
def test_a_solve_and_its_graphs(N):
    """whole CG solves (captured runs of iterations, with the inner product
    epilogue) give the same history and solution; 9 right-hand sides stay on
    the gathering kernel in FP64"""
    fd = [8, 4, 6, 8]
    U = G.random_links(R.grid(fd), R.random("march_cg"), scale=0.5)
    w = g.qcd.fermion.wilson_clover(U, ANTI, n_rhs=N)
    inv, pc = g.algorithms.inverter, g.qcd.fermion.preconditioner
    src = g.lattice(w.F_grid)
    src.data.normal_(generator=torch.Generator(device="cuda").manual_seed(5))
    got = []
    for shape, chunk in (((1, 1, 4, 1, 0), 1), (None, 1), (None, 0), (None, 0)):
        w.set_hop_shape(shape)
        w.set_iteration_chunk(chunk)
        cg = inv.cg(eps=1e-9, maxiter=500)
        x = g.eval(w.propagator(inv.preconditioned(pc.eo2_ne(), cg)) * src)
        assert cg.converged
        got.append((x.data.clone(), cg.history, cg.iterations))
    for x, hist, it in got[1:]:
        assert torch.equal(x, got[0][0]) and hist == got[0][1] and it == got[0][2]
