"""The tuner's files name the kernels that were timed: one of other kernels (an
earlier library's) is not taken, neither for a hop nor for a 16-bit one, and stays
as it is."""
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
FD = [8, 16, 16, 16]  # no other test tunes it


def solve(U, n):
    w = g.qcd.fermion.wilson_clover(U, P, n_rhs=n)
    src = g.lattice(w.F_grid)
    src.data.normal_(generator=torch.Generator(device="cuda").manual_seed(n))
    m = inv.cg_mixed(eps=1e-6, maxiter=2000, inner_storage="half")
    g(w.propagator(inv.preconditioned(pc.eo2_ne(), m)) * src)
    assert m.converged
    torch.cuda.synchronize()
    return m.inner_operator(w)


def test_files_of_earlier_kernels(tmp_path, monkeypatch):
    monkeypatch.setenv("WC_TUNE_CACHE", str(tmp_path))
    monkeypatch.delenv("WC_AUTOTUNE", raising=False)
    U = G.smooth_links(FD, 0.3, 8401)
    solve(U, 8)
    names = {f[:-5] for f in os.listdir(tmp_path)}
    hop, = [t for t in names if "_f32_" in t and t.endswith("_rhs8")]
    s16, = [t for t in names if "_f32_" in t and t.endswith("_rhs8_s16_mma")]
    assert hop.startswith("hop2_gfx950_")
    old = {}
    for tag in (hop, s16):
        tag = tag.replace("_rhs8", "_rhs16").replace("hop2_", "hop_", 1)
        old[tag] = dict(tag=tag, params=[1, 3, 5, 1, 0], ms=1.0)  # the tuner's candidates hold no such shape
        if "_s16" in tag:
            old[tag]["form"] = 1
        with open(tmp_path / (tag + ".json"), "w") as f:
            json.dump(old[tag], f)
    lo = solve(U, 16)
    assert lo.hop_shape(16) != (1, 3, 5, 1, 0)
    for tag in (hop, s16):
        assert os.path.exists(tmp_path / (tag.replace("_rhs8", "_rhs16") + ".json"))
    for tag, rec in old.items():
        assert json.load(open(tmp_path / (tag + ".json"))) == rec
