"""The next configuration on an operator that is there, from four fields or one,
on the device or the host, at any alignment: the same bits as a new operator's,
and the oracle's blocks on ragged lattices; a set_mass after it; an update in a
captured graph."""
import numpy as np
import pytest

from oracle import gauge as G
from oracle import rng as R
from oracle import wilson_clover as W

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

import gpt_amd as g  # noqa: E402
from gpt_amd import _lib, core  # noqa: E402

PARAMS = {
    "clover": dict(mass=0.1, csw_r=1.1, csw_t=0.9, xi_0=1.3, nu=0.9, isAnisotropic=True,
                   boundary_phases=[1, -1, 1j, -1]),
    "spatial": dict(mass=0.1, csw_r=1.0, csw_t=0.0, boundary_phases=[1, 1, 1, -1]),
    "open": dict(mass=0.2, csw_r=0.8, csw_t=0.8, cF=1.3, boundary_phases=[1, 1, 1, 0]),
    "plain": dict(mass=0.3, boundary_phases=[1, 1, 1, -1]),
}


def outputs(w):
    n = 2 * w.F_grid.Vh * 12
    gen = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(2 * n, generator=gen, device="cuda", dtype=w.F_grid.precision.real_dtype)
    out = []
    for op in (2001, 2002, 2005, 3001, 4001):
        y = torch.zeros_like(x)
        if _lib.load().wc_apply(w.handle, op, y.data_ptr(), x.data_ptr(), -1, core.stream_ptr()) == 0:
            out.append(y)
    assert len(out) >= 3
    return out


def links(U):
    """[4][V][3][3] on the device"""
    return torch.as_tensor(np.stack([np.asarray(u).reshape(-1, 3, 3) for u in U]), device="cuda").contiguous()


@pytest.mark.parametrize("fd", [[4, 4, 4, 4], [2, 4, 16, 4], [12, 8, 4, 6], [6, 10, 32, 2]], ids=str)
@pytest.mark.parametrize("case", list(PARAMS))
def test_every_way_in_gives_a_new_operators_bits(fd, case):
    gr = R.grid(fd)
    U1, U2 = (G.random_links(gr, R.random(t), scale=0.5) for t in ("update a", "update b"))
    f = links(U2)
    off = torch.zeros(f.numel() * 2 + 1, dtype=torch.float64, device="cuda")[1:]  # 8 bytes off
    off.copy_(torch.view_as_real(f).reshape(-1))
    host = f.cpu()
    lib, s = _lib.load(), core.stream_ptr()
    for prec, compress in ((g.double, False), (g.single, False), (g.single, True)):
        ref = g.qcd.fermion.wilson_clover(U2, PARAMS[case], precision=prec, compress_links=compress)
        expect = outputs(ref)
        ways = [
            lambda h: lib.wc_update(h, f.data_ptr(), s),
            lambda h: lib.wc_update(h, host.data_ptr(), s),
            lambda h: lib.wc_update(h, off.data_ptr(), s),
            lambda h: lib.wc_update_links(h, f[0].data_ptr(), host[1].data_ptr(), f[2].data_ptr(),
                                          off[3 * f[0].numel() * 2:].data_ptr(), s),
        ]
        w = g.qcd.fermion.wilson_clover(U1, PARAMS[case], precision=prec, compress_links=compress)
        for i, way in enumerate(ways):
            _lib.check(lib.wc_update(w.handle, links(U1).data_ptr(), s))
            if case != "open" or fd[3] > 2:  # open boundaries only: the outputs are 0 there
                assert not torch.equal(outputs(w)[0], expect[0])
            _lib.check(way(w.handle))
            _lib.check(lib.wc_set_mass(w.handle, 0.4, s))
            _lib.check(lib.wc_set_mass(w.handle, PARAMS[case]["mass"], s))
            assert all(torch.equal(a, b) for a, b in zip(outputs(w), expect)), (prec.__name__, i)
        w.release()
        ref.release()


@pytest.mark.parametrize("fd", [[2, 4, 16, 4], [12, 8, 4, 6]], ids=str)
@pytest.mark.parametrize("case", ["clover", "spatial", "open"])
def test_blocks_match_the_oracle(fd, case):
    """sums of some hundred products in FP64 on blocks of order one: 1e-13 per
    site, the bound of the operator's other tests"""
    gr = R.grid(fd)
    rng = R.random("update oracle")
    U = G.random_links(gr, rng, scale=0.8)
    src = rng.vspincolor(gr)
    ref = W.wilson_clover(U, **PARAMS[case])
    w = g.qcd.fermion.wilson_clover(U, PARAMS[case])
    for pin, cb in [(0, g.even), (1, g.odd)]:
        x = g.lattice(w.F_grid_eo)
        x.checkerboard(cb)
        x.from_numpy(src)
        masked = ref._mask(src, pin)
        for op, fn in ((w.Mooee, ref.Mooee), (w.Mooee.inv(), ref.MooeeInv)):
            want = fn(masked)
            d = np.abs(op(x).to_numpy() - want).reshape(want.shape[:4] + (-1,))
            n = np.sqrt((np.abs(want).reshape(d.shape) ** 2).sum(-1))
            assert float((np.sqrt((d**2).sum(-1)) / np.where(n > 0, n, 1)).max()) < 1e-13


def test_an_update_in_a_graph():
    """an operator without clover: nothing waits for the host, so the update can
    be captured; each replay takes the links that are there"""
    gr = R.grid([4, 4, 4, 8])
    fields = [links(G.random_links(gr, R.random(t), scale=0.5)) for t in ("g0", "g1", "g2")]
    f = fields[0].clone()
    U0 = G.random_links(gr, R.random("g0"), scale=0.5)
    w = g.qcd.fermion.wilson_clover(U0, PARAMS["plain"])
    lib = _lib.load()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        _lib.check(lib.wc_update(w.handle, f.data_ptr(), core.stream_ptr()))
    for k in (1, 2, 0, 1):
        f.copy_(fields[k])
        graph.replay()
        got = outputs(w)
        _lib.check(lib.wc_update(w.handle, fields[k].data_ptr(), core.stream_ptr()))
        assert all(torch.equal(a, b) for a, b in zip(got, outputs(w)))
        _lib.check(lib.wc_update(w.handle, fields[(k + 1) % 3].data_ptr(), core.stream_ptr()))
        assert not torch.equal(outputs(w)[0], got[0])
