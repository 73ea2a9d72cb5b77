"""The form in the tuner's files, for hops that also march through t: written as
the operator then runs, read back against the rule of sizes both ways, left open by
files without one or with an unknown one; the same solutions from all."""
import json
import os

import pytest

from oracle import gauge as G

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

import gpt_amd as g  # noqa: E402

inv = g.algorithms.inverter
pc = g.qcd.fermion.preconditioner
P = dict(mass=0.1, csw_r=1.0, csw_t=1.0, boundary_phases=[1, 1, 1, -1])


def solve(U, fd, prec, n, compress, chunk=0):
    w = g.qcd.fermion.wilson_clover(U, P, n_rhs=n, precision=prec, compress_links=compress)
    w.set_iteration_chunk(chunk)
    src = g.lattice(w.F_grid)
    src.data.normal_(generator=torch.Generator(device="cuda").manual_seed(n))
    cg = inv.cg(eps=1e-6, maxiter=12)
    x = g.eval(w.propagator(inv.preconditioned(pc.eo2_ne(), cg)) * src)
    torch.cuda.synchronize()
    return w, x.data.clone(), cg.history


# lattices that no other test tunes; the form by the rule where nothing is stored
@pytest.mark.parametrize("fd,prec,rule", [([8, 8, 16, 32], g.single, "gather"), ([8, 16, 8, 32], g.double, "gather"),
                                          ([16, 16, 16, 12], g.double, "march"), ([16, 18, 16, 12], g.single, "march")],
                         ids=str)
def test_stored_forms(fd, prec, rule, tmp_path, monkeypatch):
    monkeypatch.setenv("WC_TUNE_CACHE", str(tmp_path))
    monkeypatch.delenv("WC_AUTOTUNE", raising=False)
    U = G.smooth_links(fd, 0.3, 8301)
    w, _, _ = solve(U, fd, prec, 8, False)
    name, = [f for f in os.listdir(tmp_path) if f.endswith("_rhs8.json")]
    rec = json.load(open(tmp_path / name))
    assert rec["form"] in (0, 1) and w.hop_form() == ("march" if rec["form"] else "gather")
    # one class of counts per file: each is read once and then kept in the process
    got = []
    for cls, compress, form, want in ((16, False, 1, "march"), (16, True, 0, "gather"), (32, False, None, rule),
                                      (32, True, 7, rule)):
        tag = name[:-5].replace("_rhs8", f"_rhs{cls}")
        if compress:
            tag = tag.replace("_links18_", "_links12_")
        planted = dict(tag=tag, params=[1, 2, 8, 1, 0], ms=1.0)
        if form is not None:
            planted["form"] = form
        with open(tmp_path / (tag + ".json"), "w") as f:
            json.dump(planted, f)
        w, x, hist = solve(U, fd, prec, cls, compress)
        assert w.hop_shape() == (1, 2, 8, 1, 0) and w.hop_form() == want, (cls, compress, form)
        assert json.load(open(tmp_path / (tag + ".json"))) == planted  # neither tuned nor written
        # the other form on the same operator, after graphs of the first
        w.set_hop_form("gather" if want == "march" else "march")
        assert w.hop_form() != want
        src = g.lattice(w.F_grid)
        src.data.normal_(generator=torch.Generator(device="cuda").manual_seed(cls))
        cg = inv.cg(eps=1e-6, maxiter=12)
        y = g.eval(w.propagator(inv.preconditioned(pc.eo2_ne(), cg)) * src)
        assert torch.equal(y.data, x) and cg.history == hist and float(x.abs().max()) > 0
        w.release()
