"""The tuner where a hop takes one wave per direction, which no launch shape
changes: that form is timed, and no shape of another kernel is kept or written.
With the gathering kernel set, shapes are timed and kept as elsewhere."""
import os

import pytest

from oracle import gauge as G
from oracle import rng as R

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

import gpt_amd as g  # noqa: E402

P = dict(mass=0.1, csw_r=1.0, csw_t=1.0, boundary_phases=[1, 1, 1, -1])


@pytest.mark.parametrize("prec,n", [(g.double, 1), (g.double, 8), (g.single, 3)], ids=str)
def test_few_sites(prec, n, tmp_path, monkeypatch):
    monkeypatch.setenv("WC_TUNE_CACHE", str(tmp_path))
    fd = [6, 8, 8, 4]  # a lattice that no other test tunes
    U = G.random_links(R.grid(fd), R.random("tune_split"), scale=0.5)
    w = g.qcd.fermion.wilson_clover(U, P, precision=prec, n_rhs=n)
    default = w.hop_shape()
    assert w.hop_form() == "split"
    for by_hand in (False, True):
        if by_hand:
            w.set_hop_shape((1, 3, 8, 1, 0))
        shape, ms = w.tune_hop(reps=3)
        assert ms > 0 and shape == default == w.hop_shape() and w.hop_form() == "split"
        other = g.qcd.fermion.wilson_clover(U, dict(P, mass=0.2), precision=prec, n_rhs=n)
        assert other.hop_shape() == default and other.hop_form() == "split"
        assert os.listdir(tmp_path) == []
    w.set_hop_form("gather")
    shape, ms = w.tune_hop(reps=3)
    assert ms > 0 and w.hop_shape() == shape and w.hop_form() == "gather" and len(os.listdir(tmp_path)) == 1
    w.set_hop_form(None)
    assert w.hop_form() == "split" and w.hop_shape() == shape
    with pytest.raises(RuntimeError, match="reps"):
        w.tune_hop(reps=0)
    assert w.hop_shape() == shape
    w.release()
