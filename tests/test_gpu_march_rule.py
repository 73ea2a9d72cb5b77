"""Which hops march through t where nothing was timed or set, on both sides of each
line of the rule."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

import gpt_amd as g  # noqa: E402


@pytest.mark.parametrize("fd,prec,compress,n,want", [
    ([8, 8, 8, 8], g.double, False, 12, "march"), ([8, 8, 8, 8], g.double, True, 12, "gather"),
    ([8, 8, 8, 8], g.double, False, 13, "gather"), ([8, 8, 8, 12], g.single, False, 12, "march"),
    ([8, 8, 8, 12], g.single, False, 11, "gather"), ([8, 8, 8, 12], g.single, True, 12, "gather"),
    ([12, 12, 12, 24], g.double, False, 12, "gather"), ([14, 16, 16, 24], g.single, False, 12, "gather"),
    ([16, 16, 16, 16], g.double, False, 14, "march"), ([16, 16, 16, 16], g.double, True, 15, "gather"),
    ([16, 16, 16, 16], g.double, False, 17, "gather"), ([16, 16, 16, 16], g.double, False, 18, "march"),
    ([16, 16, 16, 16], g.single, False, 16, "march"), ([16, 16, 16, 16], g.single, False, 31, "gather"),
    ([8, 32, 32, 16], g.double, False, 16, "gather"), ([18, 16, 16, 16], g.double, False, 16, "march"),
    ([16, 16, 16, 16], g.single, False, 8, "gather"), ([16, 16, 16, 32], g.single, False, 8, "march"),
], ids=str)
def test_rule(fd, prec, compress, n, want):
    grid = g.grid(fd, g.double)
    one = torch.eye(3, dtype=torch.complex128, device="cuda").expand(grid.gsites, 3, 3).contiguous()
    w = g.qcd.fermion.wilson_clover([g.qcd.gauge.link_field(grid, one) for _ in range(4)],
                                    dict(mass=0.1, boundary_phases=[1, 1, 1, -1]), precision=prec, n_rhs=n,
                                    compress_links=compress)
    assert w.hop_form() == want
    w.release()
