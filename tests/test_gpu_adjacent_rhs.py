"""Hops of two adjacent right-hand sides per thread (one 16-byte access per
component in FP32, 8-byte in 16-bit storage) against one per thread: the same
bits for counts that two divides and that it does not, for a count of one, and
for fields aligned to one value only."""
import pytest

from oracle import gauge as G
from oracle import rng as R

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

import gpt_amd as g  # noqa: E402
from gpt_amd import _lib, core  # noqa: E402

P = dict(mass=0.1, csw_r=0.8, csw_t=0.8, boundary_phases=[1, 1, 1, -1], precision=g.single)
FD = [4, 6, 4, 8]


@pytest.fixture(scope="module")
def links():
    return G.random_links(R.grid(FD), R.random("adjacent_rhs"), scale=0.5)


def offset_field(n, dtype, shift, fill=None):
    """n values (re, im) whose address is a multiple of 16 bytes plus shift values"""
    flat = torch.zeros(2 * (n + shift), dtype=dtype, device=core.device())
    x = flat[2 * shift:]
    if fill is not None:
        x.copy_(fill)
    return x


@pytest.mark.parametrize("compress", [False, True])
@pytest.mark.parametrize("N", [1, 2, 3, 8, 13])
def test_two_per_thread_gives_the_bits_of_one(links, N, compress):
    w = g.qcd.fermion.wilson_clover(links, P, n_rhs=N, compress_links=compress)
    n = w.F_grid.Vh * 12 * N
    gen = torch.Generator(device="cuda").manual_seed(N)
    vals = torch.randn(4 * n, generator=gen, device="cuda", dtype=torch.float32)
    lib, h, s = _lib.load(), w.handle, core.stream_ptr()

    def results(rb, shift):
        out = []
        w.set_hop_shape((rb, 1, 4, 1, 1 if N > rb else 0))
        for opcode, cb, full in [(2003, 0, False), (2004, 1, False), (2001, -1, True), (2002, -1, True)]:
            m = 2 * n if full else n
            src = offset_field(m, torch.float32, shift, vals[:2 * m])
            dst = offset_field(m, torch.float32, shift)
            _lib.check(lib.wc_apply_block(h, opcode, N, dst.data_ptr(), src.data_ptr(), cb, s))
            out.append(dst.clone())
        for which in (0, 1, 2):
            src, dst = offset_field(n, torch.float32, shift, vals[:2 * n]), offset_field(n, torch.float32, shift)
            _lib.check(lib.wc_apply_mpc_block(h, 1, which, N, dst.data_ptr(), src.data_ptr(), s))
            out.append(dst.clone())
        for storage, dt in (("half", torch.float16), ("bf16", torch.bfloat16)):
            src = offset_field(n, dt, shift, vals[:2 * n].to(dt))
            dst = offset_field(n, torch.float32, shift)
            _lib.check(lib.wc_apply_mpc_block_s16(h, 1, N, _lib.STORAGE_CODES[storage], dst.data_ptr(),
                                                  src.data_ptr(), s))
            out.append(dst.clone())
        return out

    ref = results(1, 0)
    assert all(float(x.abs().sum()) > 0 for x in ref)
    for shift in (0, 1):
        for i, (a, b) in enumerate(zip(results(2, shift), ref)):
            assert torch.equal(a, b), (N, compress, shift, i)
