"""An operator taken from the pool of parked handles has the launch shapes and
forms of a new one, whatever its last owner had set."""
import gc

import pytest

from oracle import gauge as G
from oracle import rng as R

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

import gpt_amd as g  # noqa: E402

P = dict(mass=0.13, csw_r=0.9, csw_t=0.9, boundary_phases=[1, 1, 1, -1])


def test_shapes_and_forms_of_a_parked_operator():
    U = G.random_links(R.grid([4, 4, 4, 8]), R.random("pool"), scale=0.5)
    w = g.qcd.fermion.wilson_clover(U, P, n_rhs=12)
    default = {n: (w.hop_shape(n), w.hop_form(n)) for n in (1, 2, 12, 64)}
    handle = w.handle
    w.set_hop_shape((1, 3, 8, 1, 0), n_rhs=1)
    w.set_hop_shape((1, 2, 8, 1, 0))
    w.set_hop_form("march", n_rhs=64)
    w.set_hop_form("gather", n_rhs=2)
    assert all((w.hop_shape(n), w.hop_form(n)) != default[n] for n in default)
    del w
    gc.collect()
    x = g.qcd.fermion.wilson_clover(U, P, n_rhs=12)
    assert x.handle == handle
    assert {n: (x.hop_shape(n), x.hop_form(n)) for n in default} == default


def test_the_owner_keeps_its_own():
    U = G.random_links(R.grid([4, 4, 4, 8]), R.random("pool2"), scale=0.5)
    w = g.qcd.fermion.wilson_clover(U, dict(P, csw_r=0.8, csw_t=0.8))
    w.set_hop_shape((1, 3, 8, 1, 0))
    handle = w.handle
    w.suspend()
    assert w.handle == handle and w.hop_shape() == (1, 3, 8, 1, 0)
    w.suspend()
    x = g.qcd.fermion.wilson_clover(U, dict(P, csw_r=0.8, csw_t=0.8))
    assert x.handle == handle and x.hop_shape() != (1, 3, 8, 1, 0)
    x.set_hop_shape((1, 1, 8, 1, 0))
    x.suspend()
    assert w.handle == handle and w.hop_shape() not in ((1, 3, 8, 1, 0), (1, 1, 8, 1, 0))
