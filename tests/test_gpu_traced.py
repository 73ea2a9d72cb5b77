"""g.trace, pack and unpack where torch does not run the calls as they stand:
under vmap and other transforms, in traced graphs and for tensor subclasses
every value comes from torch's own operations, so that the results are those of
the plain call."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from torch.fx.experimental.proxy_tensor import make_fx  # noqa: E402
from torch.utils._python_dispatch import TorchDispatchMode  # noqa: E402

import gpt_amd as g  # noqa: E402
from gpt_amd.qcd.fermion.operator import pack, unpack  # noqa: E402

GRID = g.grid([4, 4, 4, 6], g.double)
# 144 products and sums of numbers of order 1 in another order
TOL = 148 * 2.3e-16 * 40.0


def values(seed, prec=g.double):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dt = torch.complex128 if prec is g.double else torch.complex64
    return torch.randn(GRID.gsites, 4, 4, 3, 3, generator=gen, device="cuda", dtype=dt)


def field(data, prec=g.double):
    p = g.mspincolor(g.grid(GRID.fdimensions, prec))
    p.data = data
    return p


def correlate(a, b):
    return g.trace(field(a) * g.adj(field(b))).data


def test_vmap_over_propagators():
    a, b = torch.stack([values(i) for i in range(3)]), values(7)
    want = torch.stack([correlate(x, b) for x in a])
    assert float((torch.func.vmap(correlate, (0, None))(a, b) - want).abs().max()) <= TOL
    assert float((torch.func.vmap(lambda x: correlate(x, x))(a) - torch.stack([correlate(x, x) for x in a])
                  ).abs().max()) <= TOL


@pytest.mark.parametrize("tracer", ["real", "fake", "symbolic", "jit"])
def test_a_traced_graph_holds_the_contraction(tracer):
    a, b, c, d = (values(i) for i in range(4))
    if tracer == "jit":
        f = torch.jit.trace(correlate, (a, b), check_trace=False)
    else:
        f = make_fx(correlate, tracing_mode=tracer)(a, b)
    for x, y in ((a, b), (c, d)):
        assert float((f(x, y) - correlate(x, y)).abs().max()) <= TOL


def test_modes_see_every_operation():
    class count(TorchDispatchMode):
        n = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            count.n += "mul" in str(func)
            return func(*args, **(kwargs or {}))

    a, b = values(1), values(2)
    with count():
        got = correlate(a, b)
    assert count.n == 1 and float((got - correlate(a, b)).abs().max()) <= TOL


def test_derivatives_by_transforms():
    a, t, b = values(1), values(2), values(3)
    got = torch.func.jvp(lambda x: correlate(x, b), (a,), (t,))[1]
    assert float((got - correlate(t, b)).abs().max()) <= TOL


def test_tensor_subclasses():
    class logged(torch.Tensor):
        pass

    a, b = values(1), values(2)
    got = correlate(a.as_subclass(logged), b)
    assert float((got.as_subclass(torch.Tensor) - correlate(a, b)).abs().max()) <= TOL


def test_a_traced_graph_holds_the_copies():
    def there(x, y, z):
        fs = []
        for v in (x, y, z):
            f = g.lattice(GRID)
            f.data = v
            fs.append(f)
        return pack(fs).data

    def back(p):
        f = g.lattice(g.grid(GRID.fdimensions, g.double, nrhs=3))
        f.data = p
        return [x.data for x in unpack(f)]

    def randoms(seed):
        gen = torch.Generator(device="cuda").manual_seed(seed)
        return [torch.randn(g.lattice(GRID).data.shape, generator=gen, device="cuda", dtype=torch.float64)
                for _ in range(3)]

    first, other = randoms(1), randoms(2)
    f = make_fx(there)(*first)
    assert torch.equal(f(*other), torch.cat(other, -2))
    h = make_fx(back)(torch.cat(first, -2))
    assert all(torch.equal(x, y) for x, y in zip(h(torch.cat(other, -2)), other))
