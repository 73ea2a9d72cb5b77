"""The work that programs on gpt_amd do most, as cases that can be timed and checked.

A case is a dict of plain values: ``kind`` (what is called), ``lat`` (the lattice as "XxYxZxT"), and the options of that kind:
``prec`` ("f64" / "f32"), ``links`` (18 or 12 reals stored a link), ``rhs`` (right-hand sides of one field), ``op``, ``storage``.
Lattices and counts of right-hand sides are those of bench.py and of the tests (8^4, 16^3x32, 24^3x48, 32^3x64; 1, 12 and 48),
and ragged ones between them.

  apply       an operator of the Wilson-clover object on a field: what an own solver, a force or a contraction code calls
  s16         the 16-bit normal operator that the inner solves of the mixed solver and of the server spend their time in
  update      an operator that is there gets the next gauge configuration of an ensemble and is applied
  solve       a propagator column (CG in FP64 through the even-odd normal equation)
  mixed       the production solve of many right-hand sides: FP32 inner iterations, FP64 true residual
  linalg      the vector operations of a user's own Krylov method
  correlator  the pion correlator of a propagator
  packed      the operator on a list of fields
"""
import numpy as np
import torch

import gpt_amd as g

MASS = 0.1
CSW = 1.0
PHASES = [1, 1, 1, -1]
EPS = 1e-10
# iterations of a solve at this mass on these links, for the work of a pass only
ITERATIONS = 60


def listed():
    return [
        # the smallest call: one hop of the even-odd operator on the lattice of a test run; launch and host costs
        dict(name="meooe_f64_8x8x8x8", kind="apply", op="Meooe", lat="8x8x8x8", prec="f64", links=18, rhs=1),
        # the hop of a production lattice in double precision, bench.py's headline
        dict(name="meooe_f64_32x32x32x64", kind="apply", op="Meooe", lat="32x32x32x64", prec="f64", links=18, rhs=1),
        # the adjoint of the full operator in single precision with compressed links, on a ragged lattice
        dict(name="mdag_f32_20x12x24x36", kind="apply", op="Mdag", lat="20x12x24x36", prec="f32", links=12, rhs=1),
        # the normal operator of a solve in double precision on the 12 spin-colour columns of a propagator
        dict(name="mpcne_f64_rhs12_24x24x24x48", kind="apply", op="MpcNE", lat="24x24x24x48", prec="f64", links=18,
             rhs=12),
        # the hop in single precision on the 12 columns, production lattice: the largest fields
        dict(name="meooe_f32_rhs12_32x32x32x64", kind="apply", op="Meooe", lat="32x32x32x64", prec="f32", links=18,
             rhs=12),
        # the inner operator of the mixed-precision solves with 16-bit storage
        dict(name="mpcne_half_rhs12_24x24x24x48", kind="s16", storage="half", lat="24x24x24x48", links=12, rhs=12),
        # the next configuration of an ensemble, and the first applications on it
        dict(name="update_f64_24x24x24x48", kind="update", lat="24x24x24x48", prec="f64", links=18, rhs=1),
        # one column of a point-source propagator on a small lattice: many short launches
        dict(name="solve_f64_8x8x8x8", kind="solve", lat="8x8x8x8", prec="f64", links=18, rhs=1),
        # a whole propagator's columns, mixed precision
        dict(name="mixed_rhs12_16x16x16x32", kind="mixed", lat="16x16x16x32", links=12, rhs=12),
        # a step of a user's own Krylov method
        dict(name="linalg_f64_32x32x32x64", kind="linalg", lat="32x32x32x64", prec="f64", rhs=1),
        # the measurement that follows a propagator
        dict(name="correlator_f64_24x24x24x48", kind="correlator", lat="24x24x24x48", prec="f64"),
        # twelve single fields through one batched application
        dict(name="packed_m_f64_rhs12_16x16x16x32", kind="packed", op="M", lat="16x16x16x32", prec="f64", links=18,
             rhs=12),
    ]


def draw(rng):
    """one more case of the same kinds: other lattices, counts, types and directions"""
    most = {}
    for c in listed():
        most[c["kind"]] = max(most.get(c["kind"], 0), work(c)["bytes"])
    kind = rng.choice(["apply"] * 5 + ["s16"] * 2 + ["update", "solve", "mixed", "linalg", "correlator", "packed"])
    while True:
        lat = "x".join(str(2 * int(2 ** rng.uniform(1, hi))) for hi in (4.1, 4.1, 4.1, 5.1))
        if volume(lat) % 128 or volume(lat) < 4096:
            continue
        c = dict(kind=kind, lat=lat)
        if kind not in ("s16", "mixed"):
            c["prec"] = rng.choice(["f64", "f32"])
        if kind != "correlator":
            c["rhs"] = int(2 ** rng.uniform(0, 5.6)) if kind in ("apply", "s16") else rng.choice([1, 2, 4, 5, 8, 12])
        if kind not in ("linalg", "correlator"):
            c["links"] = rng.choice([18, 12])
        if kind == "apply":
            c["op"] = rng.choice(["Meooe", "MeooeDag", "M", "Mdag", "Mooee", "MooeeInv", "Mpc", "MpcDag", "MpcNE"])
        if kind == "packed":
            c["op"] = rng.choice(["M", "Mdag"])
            c["rhs"] = rng.choice([2, 4, 5, 8, 12])
        if kind == "s16":
            c["storage"] = rng.choice(["half", "bf16"])
        if kind == "solve":
            c["prec"] = "f64"
        if kind == "update":
            c["rhs"] = 1
        if work(c)["bytes"] <= most[kind] and (kind != "solve" or volume(lat) * c["rhs"] <= 200000):
            return c


# ------------------------------------------------------------------ inputs


def dims(lat):
    return [int(x) for x in lat.split("x")]


def volume(lat):
    return int(np.prod(dims(lat)))


def generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def gauge_links(lat, gen):
    """four SU(3) fields [V, 3, 3] not far from unity, as a smooth configuration's are: 1 + 0.3 i H with H Hermitian and of
    unit variance, its first two rows made orthonormal, the third their conjugate cross product"""
    out = []
    for _ in range(4):
        n = volume(lat)
        z = torch.view_as_complex(torch.randn((n, 3, 3, 2), generator=gen, device="cuda", dtype=torch.float64))
        m = 0.3j * 0.5 * (z + z.conj().transpose(1, 2)) + torch.eye(3, device="cuda", dtype=torch.complex128)
        a = m[:, 0] / m[:, 0].abs().square().sum(1, keepdim=True).sqrt()
        b = m[:, 1] - (a.conj() * m[:, 1]).sum(1, keepdim=True) * a
        b = b / b.abs().square().sum(1, keepdim=True).sqrt()
        c = torch.stack([a[:, 1] * b[:, 2] - a[:, 2] * b[:, 1], a[:, 2] * b[:, 0] - a[:, 0] * b[:, 2],
                         a[:, 0] * b[:, 1] - a[:, 1] * b[:, 0]], 1).conj()
        out.append(torch.stack([a, b, c], 1).contiguous())
    return out


def real_type(case):
    return torch.float64 if case.get("prec", "f64") == "f64" else torch.float32


def field_values(case, gen, parities, dtype=None):
    """Gaussian spinors in the order of a field's storage"""
    n = volume(case["lat"]) // 2
    shape = (n // 64, 12, 64, case.get("rhs", 1), 2)
    return torch.randn((2,) + shape if parities == 2 else shape, generator=gen, device="cuda",
                       dtype=dtype or real_type(case))


def point_values(case):
    """right-hand side r: the unit vector of component r % 12 at the origin"""
    n = volume(case["lat"]) // 2
    x = torch.zeros((2, n // 64, 12, 64, case["rhs"], 2), device="cuda", dtype=torch.float64)
    for r in range(case["rhs"]):
        x[0, 0, r % 12, 0, r, 0] = 1.0
    return x


def propagator_values(case, gen):
    """[V, 4, 4, 3, 3], decaying with the distance in time from the source"""
    t = torch.arange(dims(case["lat"])[3], device="cuda", dtype=torch.float64)
    fall = torch.exp(-0.3 * torch.minimum(t, t.numel() - t)).repeat_interleave(volume(case["lat"]) // t.numel())
    z = torch.randn((volume(case["lat"]), 144, 2), generator=gen, device="cuda", dtype=real_type(case))
    z.mul_(fall.to(z.dtype)[:, None, None])
    return torch.view_as_complex(z).reshape(-1, 4, 4, 3, 3)


def draw_inputs(case, seed):
    """everything that a state is made from: plain tensors, from the seed alone"""
    gen = generator(seed)
    kind = case["kind"]
    if kind == "linalg":
        return dict(x=field_values(case, gen, 2), y=field_values(case, gen, 2))
    if kind == "correlator":
        return dict(prop=propagator_values(case, gen))
    i = dict(U=gauge_links(case["lat"], gen))
    if kind == "apply":
        i["x"] = field_values(case, gen, 2 if case["op"] in ("M", "Mdag") else 1)
    elif kind == "s16":
        i["x"] = field_values(case, gen, 1, torch.float32).to(
            torch.float16 if case["storage"] == "half" else torch.bfloat16)
    elif kind == "update":
        i["x"], i["y"] = field_values(case, gen, 2), field_values(case, gen, 1)
    elif kind == "solve":
        i["x"] = point_values(case)
    else:
        i["x"] = field_values(case, gen, 2)
    return i


# ---------------------------------------------------- what a program holds


def operator(case, U, precision, n_rhs):
    grid = g.grid(dims(case["lat"]), g.double)
    links = [g.qcd.gauge.link_field(grid, u) for u in U]
    return g.qcd.fermion.wilson_clover(
        links, dict(mass=MASS, csw_r=CSW, csw_t=CSW, boundary_phases=PHASES, precision=precision,
                    compress_links=case["links"] == 12, n_rhs=n_rhs))


def field(grid, values, cb=None):
    x = g.lattice(grid)
    x.data.copy_(values)
    if cb is not None:
        x.checkerboard(cb)
    return x


def prepare(case, seed):
    i, kind = draw_inputs(case, seed), case["kind"]
    s = dict(kind=kind)
    precision = g.double if case.get("prec", "f64") == "f64" else g.single
    if kind == "linalg":
        grid = g.grid(dims(case["lat"]), precision, nrhs=case["rhs"])
        s.update(x=field(grid, i["x"]), y=field(grid, i["y"]), z=g.lattice(grid))
        return s
    if kind == "correlator":
        s["prop"] = g.mspincolor(g.grid(dims(case["lat"]), precision))
        s["prop"].data.copy_(i["prop"])
        return s
    pc, inv = g.qcd.fermion.preconditioner, g.algorithms.inverter
    if kind == "s16":
        s.update(w=operator(case, i["U"], g.single, case["rhs"]), x=i["x"], storage=case["storage"])
        return s
    if kind == "mixed":
        # the solver makes its own FP32 operator, on 12-real links by default
        w = operator(dict(case, links=18), i["U"], g.double, case["rhs"])
        solver = inv.cg_mixed(eps=EPS, inner_compress_links=case["links"] == 12)
        s.update(w=w, slv=w.propagator(inv.preconditioned(pc.eo2_ne(), solver)), src=field(w.F_grid, i["x"]))
        return s
    w = operator(case, i["U"], precision, case["rhs"])
    s["w"] = w
    if kind == "solve":
        s["slv"] = w.propagator(inv.preconditioned(pc.eo2_ne(), inv.cg(eps=EPS, maxiter=1000)))
        s["src"] = field(w.F_grid, i["x"])
    elif kind == "packed":
        one = w.F_grid.single_rhs()
        s["srcs"] = [field(one, i["x"][..., r:r + 1, :]) for r in range(case["rhs"])]
        s["op"] = w.packed() if case["op"] == "M" else w.adj().packed()
    elif kind == "update":
        grid = g.grid(dims(case["lat"]), g.double)
        s["U"] = [g.qcd.gauge.link_field(grid, u) for u in i["U"]]
        s["psi"], s["half"] = field(w.F_grid, i["x"]), field(w.F_grid_eo, i["y"], g.odd)
    else:
        schur = pc.eo2_ne()(w)
        s["op"] = {"M": w, "Mdag": w.adj(), "Meooe": w.Meooe, "MeooeDag": w.Meooe.adj(), "Mooee": w.Mooee,
                   "MooeeInv": w.Mooee.inv(), "Mpc": schur.Mpc_schur, "MpcDag": schur.Mpc_schur.adj(),
                   "MpcNE": schur.Mpc}[case["op"]]
        if case["op"] in ("M", "Mdag"):
            s["src"] = field(w.F_grid, i["x"])
        else:
            s["src"] = field(w.F_grid_eo, i["x"], g.odd)
    return s


# -------------------------------------------------------------------- pass


def run(s):
    kind = s["kind"]
    if kind == "apply":
        return s["op"](s["src"]).data
    if kind == "s16":
        return s["w"].mpc_ne_s16(s["x"], 1, s["storage"])
    if kind == "update":
        s["w"].update(s["U"])
        return dict(m=s["w"](s["psi"]).data, inv=s["w"].Mooee.inv()(s["half"]).data)
    if kind in ("solve", "mixed"):
        return g(s["slv"] * s["src"]).data
    if kind == "linalg":
        n2 = g.axpy_norm2(s["z"], 0.7 - 0.2j, s["x"], s["y"])
        ip = g.inner_product(s["x"], s["z"])
        nx = g.norm2(s["x"])
        return dict(z=s["z"].data, n2=n2, ip=np.complex128(ip), nx=nx)
    if kind == "correlator":
        return np.array(g.slice(g.trace(s["prop"] * g.adj(s["prop"])), 3))
    return [x.data for x in s["op"](s["srcs"])]


# -------------------------------------------------------------------- work


def work(case):
    """bytes and operations that a pass cannot do without; counts of a site: a link 8 times a hop (4 links of each of the two
    sites of a pair), a clover block or its inverse 72 reals, a spinor 24; a hop 1320, a clover product 552 operations"""
    v, n, kind = volume(case["lat"]), case.get("rhs", 1), case["kind"]
    h = v // 2
    r = 8 if case.get("prec", "f64") == "f64" else 4
    links = h * 8 * case.get("links", 18) * r
    clover, spinor = h * 72 * r, h * 24 * n * r
    hop, site = h * 1320 * n, h * 552 * n
    if kind == "apply":
        return {
            "Meooe": dict(bytes=links + 2 * spinor, flops=hop),
            "MeooeDag": dict(bytes=links + 2 * spinor, flops=hop),
            "Mooee": dict(bytes=clover + 2 * spinor, flops=site),
            "MooeeInv": dict(bytes=clover + 2 * spinor, flops=site),
            "M": dict(bytes=links + 2 * clover + 4 * spinor, flops=2 * (hop + site)),
            "Mdag": dict(bytes=links + 2 * clover + 4 * spinor, flops=2 * (hop + site)),
            "Mpc": dict(bytes=links + 2 * clover + 2 * spinor, flops=2 * (hop + site)),
            "MpcDag": dict(bytes=links + 2 * clover + 2 * spinor, flops=2 * (hop + site)),
            "MpcNE": dict(bytes=links + 2 * clover + 2 * spinor, flops=4 * (hop + site)),
        }[case["op"]]
    if kind == "s16":
        return dict(bytes=h * (8 * case["links"] * 4 + 2 * 72 * 4 + 24 * n * (2 + 4)), flops=4 * (hop + site))
    if kind == "update":
        # the links in, their stored form, the clover blocks and their inverses, and the two applications
        return dict(bytes=v * 72 * 8 + 2 * links + 4 * clover + links + 3 * clover + 6 * spinor,
                    flops=v * 6 * 5600 + 2 * (hop + site) + site)
    if kind == "solve":
        # every iteration reads links, inverse blocks and a search direction, and writes the next
        return dict(bytes=ITERATIONS * (links + 2 * clover + 8 * spinor), flops=ITERATIONS * 4 * (hop + site))
    if kind == "mixed":
        return dict(bytes=ITERATIONS * h * 4 * (8 * case["links"] + 2 * 72 + 8 * 24 * n),
                    flops=ITERATIONS * 4 * (hop + site))
    if kind == "linalg":
        return dict(bytes=2 * 3 * spinor, flops=v * n * 24 * 8)
    if kind == "correlator":
        return dict(bytes=v * 144 * 2 * r + v * 16, flops=v * 144 * 8)
    # packed: the list in and out
    return dict(bytes=links + 2 * clover + 4 * spinor, flops=2 * (hop + site))


# ------------------------------------------------- the same in 64 bits, plain


def matmul3(a, b):
    return (a[..., :, :, None] * b[..., None, :, :]).sum(-2)


def dagger(a):
    return a.conj().transpose(-1, -2)


# (1 - s gamma_mu) psi with gamma in the chiral basis: gamma psi has the component `phase` times psi[`from`]
GAMMA = [((3, 2, 1, 0), (1j, 1j, -1j, -1j)), ((3, 2, 1, 0), (-1, 1, 1, -1)), ((2, 3, 0, 1), (1j, -1j, -1j, 1j)),
         ((2, 3, 0, 1), (1, 1, 1, 1))]


class plain_operator:
    """the Wilson-clover operator on natural fields [T, Z, Y, X, 4, 3, N] in complex128"""

    def __init__(self, lat, U):
        self.dims = dims(lat)
        self.shape = tuple(reversed(self.dims))
        self.U0 = [u.reshape(self.shape + (3, 3)) for u in U]
        self.U = []
        for mu in range(4):
            u = self.U0[mu].clone()
            u.select(3 - mu, self.dims[mu] - 1).mul_(PHASES[mu])
            self.U.append(u)
        self.diag = MASS + 4.0
        self.build_clover()

    def build_clover(self):
        gam = []
        for perm, phase in GAMMA:
            m = np.zeros((4, 4), complex)
            for i in range(4):
                m[i, perm[i]] = phase[i]
            gam.append(m)
        # chiral blocks [2][..., 2, 3, 2, 3]
        A = [torch.zeros(self.shape + (2, 3, 2, 3), device="cuda", dtype=torch.complex128) for _ in range(2)]
        at = lambda u, *steps: torch.roll(u, [-d for _, d in steps], [3 - m for m, _ in steps])  # noqa: E731
        for mu in range(4):
            for nu in range(mu + 1, 4):
                Um, Un = self.U0[mu], self.U0[nu]
                up = matmul3(matmul3(at(Un, (mu, 1)), dagger(at(Um, (nu, 1)))), dagger(Un))
                down = matmul3(dagger(matmul3(at(Um, (nu, -1)), at(Un, (nu, -1), (mu, 1)))), at(Un, (nu, -1)))
                v = up - down
                q = matmul3(Um, v) + at(matmul3(v, Um), (mu, -1))
                F = 0.125 * (q - dagger(q))
                s = 0.5 * (gam[mu] @ gam[nu] - gam[nu] @ gam[mu])
                for ch in range(2):
                    for a in range(2):
                        for b in range(2):
                            z = complex(s[2 * ch + a, 2 * ch + b])
                            if z:
                                A[ch][..., a, :, b, :] += (-0.5 * CSW * z) * F
        self.A, self.Ainv = [], []
        for ch in range(2):
            m = A[ch].reshape(self.shape + (6, 6))
            m = m + self.diag * torch.eye(6, device="cuda", dtype=torch.complex128)
            self.A.append(m)
            inv = m.clone()  # Gauss-Jordan in place; the blocks are near the positive diagonal
            for k in range(6):
                p = 1.0 / inv[..., k, k]
                row = inv[..., k, :] * p[..., None]
                col = inv[..., :, k].clone()
                inv = inv - col[..., :, None] * row[..., None, :]
                inv[..., k, :] = row
                inv[..., :, k] = -col * p[..., None]
                inv[..., k, k] = p
            self.Ainv.append(inv)

    def site(self, blocks, x):
        """the 6x6 blocks on a spinor field"""
        out = torch.empty_like(x)
        for ch in range(2):
            v = x[..., 2 * ch:2 * ch + 2, :, :].flatten(-3, -2)
            o = blocks[ch][..., :, 0, None] * v[..., None, 0, :]
            for k in range(1, 6):
                o += blocks[ch][..., :, k, None] * v[..., None, k, :]
            out[..., 2 * ch:2 * ch + 2, :, :] = o.unflatten(-2, (2, 3))
        return out

    def hop(self, x, dag=False):
        out = torch.zeros_like(x)
        for mu in range(4):
            perm, phase = GAMMA[mu]
            for fb in (1, -1):
                s = fb * (-1 if dag else 1)
                y = torch.roll(x, -fb, 3 - mu)
                u = self.U[mu] if fb == 1 else dagger(torch.roll(self.U[mu], 1, 3 - mu))
                up = [y[..., i, :, :] - s * phase[i] * y[..., perm[i], :, :] for i in range(2)]
                for i in range(2):
                    h = u[..., :, 0, None] * up[i][..., None, 0, :]
                    h += u[..., :, 1, None] * up[i][..., None, 1, :]
                    h += u[..., :, 2, None] * up[i][..., None, 2, :]
                    out[..., i, :, :] -= 0.5 * h
                    # (1 - s gamma) psi: its lower component perm[i] is -s phase[perm[i]] times the upper one
                    out[..., perm[i], :, :] += (0.5 * s * phase[perm[i]]) * h
        return out

    def m(self, x, dag=False):
        return self.hop(x, dag) + self.site(self.A, x)


def site_order(lat, parity):
    """natural index of each half-site of a parity"""
    L = dims(lat)
    h = torch.arange(volume(lat) // 2, device="cuda")
    row = h // (L[0] // 2)
    odd = (row % L[1] + row // L[1] % L[2] + row // (L[1] * L[2]) + parity) % 2
    return 2 * h + odd


def to_natural(lat, halves):
    """{parity: stored values} -> [T, Z, Y, X, 4, 3, N]"""
    n = next(iter(halves.values())).shape[-2]
    out = torch.zeros((volume(lat), 12, n), device="cuda", dtype=torch.complex128)
    for p, x in halves.items():
        z = torch.view_as_complex(x.to(torch.float64).contiguous())
        out[site_order(lat, p)] = z.permute(0, 2, 1, 3).reshape(-1, 12, n)
    return out.reshape(tuple(reversed(dims(lat))) + (4, 3, n))


def to_stored(lat, x, parity):
    """[T, Z, Y, X, 4, 3, N] -> stored values of a parity"""
    n = x.shape[-1]
    half = x.reshape(-1, 12, n)[site_order(lat, parity)]
    return torch.view_as_real(half.reshape(-1, 64, 12, n).permute(0, 2, 1, 3).contiguous())


def both(lat, x):
    return torch.stack([to_stored(lat, x, 0), to_stored(lat, x, 1)])


def only(lat, x, parity):
    """x on the sites of a parity, zero on the others"""
    keep = torch.zeros(volume(lat), device="cuda", dtype=torch.float64)
    keep[site_order(lat, parity)] = 1.0
    return x * keep.reshape(x.shape[:4] + (1, 1, 1))


def plain_solve(D, b):
    """M^-1 b for every right-hand side by BiCGStab, restarted until the residual no longer falls"""
    dot = lambda u, v: (u.conj() * v).sum((0, 1, 2, 3, 4, 5))  # noqa: E731
    x = torch.zeros_like(b)
    bb = dot(b, b).real
    for _ in range(4):
        r = b - D.m(x)
        if float((dot(r, r).real / bb).max()) < 1e-28:
            break
        r0, p = r.clone(), r.clone()
        rho = dot(r0, r)
        for _ in range(300):
            v = D.m(p)
            alpha = rho / dot(r0, v)
            s = r - alpha * v
            t = D.m(s)
            omega = dot(t, s) / dot(t, t)
            x += alpha * p + omega * s
            r = s - omega * t
            if float((dot(r, r).real / bb).max()) < 1e-29:
                break
            new = dot(r0, r)
            p = r + (new / rho) * (alpha / omega) * (p - omega * v)
            rho = new
    return x


def exact(case, seed):
    kind, lat = case["kind"], case["lat"]
    i = draw_inputs(case, seed)
    if kind == "linalg":
        x = torch.view_as_complex(i["x"].double())
        z = (0.7 - 0.2j) * x + torch.view_as_complex(i["y"].double())
        dot = lambda u, v: complex((u.conj() * v).sum().cpu())  # noqa: E731
        # of a field of several right-hand sides, norm2 gives one value each
        nx = [float(v) for v in x.abs().square().flatten(0, -2).sum(0).cpu()]
        return dict(z=torch.view_as_real(z), n2=dot(z, z).real, ip=np.complex128(dot(x, z)),
                    nx=nx if case["rhs"] > 1 else nx[0])
    if kind == "correlator":
        p = i["prop"].to(torch.complex128)
        return p.abs().square().reshape(dims(lat)[3], -1).sum(1).cpu().numpy().astype(np.complex128)
    D = plain_operator(lat, i["U"])
    if kind in ("solve", "mixed"):
        return both(lat, plain_solve(D, to_natural(lat, {0: i["x"][0], 1: i["x"][1]})))
    if kind == "packed":
        out = both(lat, D.m(to_natural(lat, {0: i["x"][0], 1: i["x"][1]}), case["op"] == "Mdag"))
        return [out[..., r:r + 1, :].contiguous() for r in range(case["rhs"])]
    if kind == "update":
        half = to_natural(lat, {1: i["y"]})
        return dict(m=both(lat, D.m(to_natural(lat, {0: i["x"][0], 1: i["x"][1]}))),
                    inv=to_stored(lat, D.site(D.Ainv, half), 1))
    op = case.get("op", "MpcNE")
    if op in ("M", "Mdag"):
        return both(lat, D.m(to_natural(lat, {0: i["x"][0], 1: i["x"][1]}), op == "Mdag"))
    x = to_natural(lat, {1: i["x"]})
    if op in ("Meooe", "MeooeDag"):
        return to_stored(lat, D.hop(x, op == "MeooeDag"), 0)
    if op in ("Mooee", "MooeeInv"):
        return to_stored(lat, D.site(D.A if op == "Mooee" else D.Ainv, x), 1)
    # 1 - Meooe A^-1 Meooe A^-1 on the odd sites, and its adjoint
    there = lambda v: v - only(lat, D.hop(D.site(D.Ainv, D.hop(D.site(D.Ainv, v)))), 1)  # noqa: E731
    back = lambda v: v - only(lat, D.site(D.Ainv, D.hop(D.site(D.Ainv, D.hop(v, True)), True)), 1)  # noqa: E731
    if op == "Mpc":
        x = there(x)
    elif op == "MpcDag":
        x = back(x)
    else:
        x = back(there(x))
    return to_stored(lat, x, 1)
