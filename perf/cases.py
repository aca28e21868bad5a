"""Performance cases of the spectral-element hot path.

Each case is a call that a user of the library makes, on the shapes it is used
for: Helmholtz / Poisson solves alone and batched, in the precisions and with
the preconditioners the library offers, the operator apply, semi-Lagrangian
advection of both orders, whole QG channel steps and a served two-layer
stream.  listed() holds the fixed cases, draw() gives more of the same ranges,
prepare() builds what a program holds before the call, run() makes the call,
work() states the bytes and flops it cannot do without, and exact() computes
the same outputs in 64-bit numpy from the definitions alone.
"""
import math

import numpy as np
import torch

import se_amd

TWO_PI = 2.0 * math.pi

# boundary layouts: name -> (periodic x, periodic y, (bottom, top, left, right) walls)
BCS = {
    "periodic": ((1, 1), (0, 0, 0, 0)),
    "channel": ((1, 0), (1, 1, 0, 0)),
    "box": ((0, 0), (1, 1, 1, 1)),
    "floor": ((0, 0), (1, 0, 0, 0)),
}
# solver variants: name -> (precision, preconditioner)
SOLVERS = {
    "fp64": (se_amd.PREC_FP64, se_amd.PC_DEFAULT),
    "fp64_fdm": (se_amd.PREC_FP64, se_amd.PC_FDM),
    "fp32_ir": (se_amd.PREC_FP32_IR, se_amd.PC_DEFAULT),
    "fp64_fp32c": (se_amd.PREC_FP64_FP32C, se_amd.PC_FDM),
    "fp64_bf16c": (se_amd.PREC_FP64_BF16C, se_amd.PC_FDM),
    "fp32_jacobi": (se_amd.PREC_FP32_IR, se_amd.PC_JACOBI),
}


def _solve(name, ex, ey, p, bc, solver, c_mass, c_lap=1.0, detj=1, null=False):
    return dict(name=name, kind="solve", ex=ex, ey=ey, p=p, bc=bc, solver=solver, c_mass=c_mass, c_lap=c_lap,
                detj=detj, null=null)


def listed():
    return [
        # the smallest solve: doubly periodic Poisson, 1024 unknowns, default options
        _solve("poisson_8x8_p4", 8, 8, 4, "periodic", "fp64", 0.0, -1.0, 0, True),
        # the inversion of a one-layer QG channel model, default options
        _solve("channel_32x32_p6", 32, 32, 6, "channel", "fp64", -100.0, -1.0, 0),
        # one large Helmholtz problem with the reference's algorithm (FP64 Jacobi-PCG) ...
        _solve("helmholtz_128x128_p8_jacobi", 128, 128, 8, "periodic", "fp64", 100.0),
        # ... and with fast diagonalisation
        _solve("helmholtz_128x128_p8_fdm", 128, 128, 8, "periodic", "fp64_fdm", 100.0),
        # an ordinary closed box with element counts that are no powers of two
        _solve("box_45x29_p5_fp32", 45, 29, 5, "box", "fp32_ir", 10.0),
        # the ensemble: 512 uneven periodic problems in one batch
        dict(name="ensemble_512", kind="batch", count=512, emin=8, emax=64, pow2=True, bc="periodic",
             solver="fp64_bf16c"),
        # a small batch of ragged channel problems in the batch's default precision
        dict(name="batch_24_channel", kind="batch", count=24, emin=10, emax=50, pow2=False, bc="channel",
             solver="fp32_ir"),
        # one operator product, as an outer iteration of the caller's own makes it
        dict(name="apply_61x47_p7", kind="apply", ex=61, ey=47, p=7, bc="box", c_mass=3.0, c_lap=1.0, detj=1),
        # velocities and second-order advection of one field: the transport part of a model step
        dict(name="advect2_96x96_p6", kind="advect", ex=96, ey=96, p=6, bc="channel", order=2, dofs=1),
        # first-order advection of a vector field with departure elements, closed box
        dict(name="advect1_29x17_p5", kind="advect", ex=29, ey=17, p=5, bc="box", order=1, dofs=2),
        # three steps of the one-layer channel model with drag, default options, host state in and out
        dict(name="qg_channel_32_p6", kind="qg", ex=32, ey=32, p=6, solver="fp64", steps=3, drag=0.1),
        # a served two-layer stream: requests of several sizes and lengths at once
        dict(name="stream_8", kind="stream", count=8, emin=16, emax=48, p=6, smax=5, solver="fp32_ir"),
    ]


def _logint(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    """One more case of the listed ranges."""
    kind = rng.choice(["solve", "solve", "solve", "batch", "apply", "advect", "advect", "qg", "stream"])
    if kind == "solve":
        solver = rng.choice(["fp64", "fp64", "fp64_fdm", "fp32_ir", "fp64_fp32c", "fp64_bf16c", "fp32_jacobi"])
        jac = solver in ("fp64", "fp32_jacobi")
        bc = rng.choice(sorted(BCS))
        return dict(kind="solve", ex=_logint(rng, 6, 64 if jac else 120), ey=_logint(rng, 6, 64 if jac else 120),
                    p=rng.randint(3, 8), bc=bc, solver=solver, c_mass=10.0 ** rng.uniform(0.0, 3.0), c_lap=1.0,
                    detj=1, null=False)
    if kind == "batch":
        return dict(kind="batch", count=_logint(rng, 4, 128), emin=8, emax=_logint(rng, 16, 56), pow2=False,
                    bc=rng.choice(["periodic", "channel", "box"]),
                    solver=rng.choice(["fp64_bf16c", "fp64_fp32c", "fp64_fdm", "fp32_ir"]))
    if kind == "apply":
        return dict(kind="apply", ex=_logint(rng, 8, 128), ey=_logint(rng, 8, 128), p=rng.randint(2, 8),
                    bc=rng.choice(sorted(BCS)), c_mass=rng.uniform(0.5, 100.0), c_lap=1.0, detj=rng.randint(0, 1))
    if kind == "advect":
        return dict(kind="advect", ex=_logint(rng, 8, 96), ey=_logint(rng, 8, 96), p=rng.randint(3, 8),
                    bc=rng.choice(["periodic", "channel", "box"]), order=rng.randint(1, 2), dofs=rng.randint(1, 3))
    if kind == "qg":
        e = _logint(rng, 8, 40)
        return dict(kind="qg", ex=e, ey=max(6, e - rng.randint(0, 5)), p=rng.randint(4, 7),
                    solver=rng.choice(["fp64", "fp64_fdm", "fp32_ir"]), steps=rng.randint(1, 4),
                    drag=rng.choice([0.0, 0.1]))
    return dict(kind="stream", count=rng.randint(2, 8), emin=12, emax=_logint(rng, 20, 48), p=rng.randint(4, 7),
                smax=rng.randint(2, 5), solver=rng.choice(["fp32_ir", "fp64_bf16c"]))


# ---------------------------------------------------------------------------
# inputs: everything random comes from numpy's generator, from the seed alone

_gll_cache = {}


def gll(p):
    """GLL abscissae, weights and differentiation matrix D[i][j] = l_j'(x_i)."""
    if p not in _gll_cache:
        c = np.zeros(p + 1)
        c[p] = 1.0
        P = np.polynomial.legendre
        x = np.concatenate([[-1.0], np.sort(np.real(P.legroots(P.legder(c)))), [1.0]])
        for _ in range(3):  # Newton polish of the inner roots of P_p'
            x[1:-1] -= P.legval(x[1:-1], P.legder(c)) / P.legval(x[1:-1], P.legder(c, 2))
        L = P.legval(x, c)
        D = np.zeros((p + 1, p + 1))
        for i in range(p + 1):
            for j in range(p + 1):
                if i != j:
                    D[i, j] = L[i] / (L[j] * (x[i] - x[j]))
        D -= np.diag(D.sum(1))
        _gll_cache[p] = (x, 2.0 / (p * (p + 1) * L * L), D)
    return _gll_cache[p]


def _line(ne, p, lo, hi):
    """Vertex coordinates of one direction."""
    dx = (hi - lo) / ne
    i = np.arange(ne * p + 1)
    return lo + (i // p) * dx + (gll(p)[0][i % p] + 1.0) / 2.0 * dx


def _domain(case):
    """The box of a case: [0, 2 pi]^2 for the Helmholtz problems, the unit square otherwise."""
    return TWO_PI if case["kind"] in ("solve", "batch", "apply") else 1.0


def _smooth(rng, X, Y, L, bc, kmax):
    """A random field on the lines X, Y with spectrum |k|^-1.5 up to kmax, unit
    mean square: periodic, or a mirrored spectrum (sines and cosines of half
    wave numbers) across walls."""
    k = np.arange(1, max(2, kmax + 1))
    per = BCS[bc][0]

    def basis(Z, periodic):
        s = (TWO_PI if periodic else math.pi) / L
        return np.concatenate([np.ones((len(Z), 1)), np.cos(s * np.outer(Z, k)), np.sin(s * np.outer(Z, k))], 1)

    kk = np.concatenate([[0.0], k, k])
    amp = (1.0 + kk[:, None] ** 2 + kk[None, :] ** 2) ** -0.75
    amp[0, 0] = 0.0
    f = basis(Y, per[1]) @ (rng.standard_normal(amp.shape) * amp) @ basis(X, per[0]).T
    return np.ascontiguousarray(f / math.sqrt(np.mean(f * f)))


def _vortices(rng, X, Y, count, walls):
    """Gaussian vortices on the unit square (x-periodic), zero on the walls."""
    q = np.zeros((len(Y), len(X)))
    for cx, cy, r, a in zip(rng.random(count), rng.random(count), 0.03 + 0.06 * rng.random(count),
                            rng.standard_normal(count)):
        dx = X - cx
        dx -= np.round(dx)
        q += a * np.exp(-((Y - cy) ** 2)[:, None] / (r * r)) * np.exp(-(dx * dx)[None, :] / (r * r))
    return q * np.sin(math.pi * Y)[:, None] if walls else q


def _members(case):
    """Sizes, orders and coefficients of a batch: part of the case, not of the seed."""
    rng = np.random.default_rng(case["count"] * 1000003 + case["emax"] * 101 + len(case["bc"]))
    out = []
    for _ in range(case["count"]):
        if case["pow2"]:
            ex = ey = int(case["emin"] * 2 ** rng.integers(0, int(math.log2(case["emax"] // case["emin"])) + 1))
            p = int(rng.choice([4, 6, 8]))
        else:
            ex, ey = (int(round(case["emin"] * (case["emax"] / case["emin"]) ** u)) for u in rng.random(2))
            p = int(rng.integers(3, 9))
        out.append(dict(kind="batch", ex=ex, ey=ey, p=p, bc=case["bc"], c_mass=float(10.0 ** rng.uniform(0.0, 3.0)),
                        c_lap=1.0, detj=1))
    return out


def _layout(members):
    """The solutions of a batch lie back to back, one array per order, each from
    a multiple of 32 values on: (array, first value) of every member, array sizes."""
    orders = sorted({m["p"] for m in members})
    sizes = [0] * len(orders)
    where = []
    for m in members:
        k = orders.index(m["p"])
        where.append((k, sizes[k]))
        sizes[k] += (math.prod(_free_shape(m)) + 31) // 32 * 32
    return where, sizes


def _requests(case):
    """Sizes and step counts of a served stream: part of the case, not of the seed."""
    rng = np.random.default_rng(case["count"] * 7919 + case["emax"])
    e = [int(round(case["emin"] * (case["emax"] / case["emin"]) ** u)) for u in rng.random(case["count"])]
    return [dict(kind="stream", ex=m, ey=m, p=case["p"], bc="channel", steps=int(s))
            for m, s in zip(e, rng.integers(1, case["smax"] + 1, case["count"]))]


def _host_inputs(case, seed):
    """The host arrays of one problem (numpy, the field layout [nV1][nV0] flattened by the caller)."""
    rng = np.random.default_rng([seed & 0x7FFFFFFF, case["ex"], case["ey"], case["p"]])
    L = _domain(case)
    X, Y = _line(case["ex"], case["p"], 0.0, L), _line(case["ey"], case["p"], 0.0, L)
    kind = case["kind"]
    if kind in ("solve", "batch", "apply"):
        bc = case["bc"]
        kmax = min(32, max(2, case["ex"] * case["p"] // 4), max(2, case["ey"] * case["p"] // 4))
        d = dict(rhs=_smooth(rng, X, Y, L, bc, kmax))
        wall = np.zeros_like(d["rhs"])
        if kind == "solve" and bc != "periodic":
            g = _smooth(rng, X, Y, L, bc, 3)
            wall[_wall_mask(case)] = g[_wall_mask(case)]
        d["wall"] = wall
        if kind == "apply":
            d["x"] = rng.standard_normal(_free_shape(case)).ravel()
        return d
    if kind == "advect":
        walls = case["bc"] != "periodic"
        psi = _vortices(rng, X, Y, 12, walls) if case["bc"] != "box" else \
            _vortices(rng, X, Y, 12, True) * np.sin(math.pi * X)[None, :]
        psip = psi * 0.97 + 0.03 * np.roll(psi, 1, 0) * (np.sin(math.pi * Y)[:, None] if walls else 1.0)
        q = np.stack([_smooth(rng, X, Y, L, case["bc"], 12) for _ in range(case["dofs"])], -1)
        qp = np.stack([_smooth(rng, X, Y, L, case["bc"], 12) for _ in range(case["dofs"])], -1) * 0.1 + q
        dt = _cfl(case, _genvel(case, psi))
        return dict(psi=psi, psip=psip, q=q, qp=qp, dt=dt)
    psi = [_vortices(rng, X, Y, 12, True) for _ in range(2 if kind == "stream" else 1)]
    om = [_vortices(rng, X, Y, 12, True) * 50.0 for _ in psi]
    dt = min(_cfl(case, _genvel(case, p)) for p in psi)
    return dict(psi=psi, om=om, dt=dt)


# ---------------------------------------------------------------------------
# the calls


def _mesh(ctx, case):
    per, bc = BCS[case.get("bc", "channel")]
    L = _domain(case)
    return se_amd.Mesh(ctx, (case["ex"], case["ey"]), case["p"], (0.0, 0.0), (L, L), per, bc)


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a).ravel()).cuda()


def prepare(case, seed):
    if case["kind"] == "stream":
        prec, pc = SOLVERS[case["solver"]]
        reqs = []
        for i, r in enumerate(_requests(case)):
            d = _host_inputs(r, seed * 64 + i)
            req = dict(nEls=(r["ex"], r["ey"]), N=r["p"], lo=(0.0, 0.0), hi=(1.0, 1.0), periodic=(1, 0),
                       bc=(1, 1, 0, 0), F1=200.0, F2=200.0, beta=1.0, steps=r["steps"])
            reqs.append((req, [d["psi"][0].ravel(), d["om"][0].ravel(), d["psi"][1].ravel(), d["om"][1].ravel()],
                         d["dt"]))
        return dict(case=case, server=se_amd.Server(0, precision=prec, preconditioner=pc), reqs=reqs)
    ctx = se_amd.Context(0)
    st = dict(case=case, ctx=ctx)
    lib = se_amd.lib()
    if case["kind"] == "batch":
        members = _members(case)
        where, sizes = _layout(members)
        st["out"] = [torch.zeros(n, dtype=torch.float64, device="cuda") for n in sizes]
        st["helms"], st["f"], st["xp"] = [], [], []
        for i, mc in enumerate(members):
            mesh = _mesh(ctx, mc)
            h = se_amd.Helm(mesh, mc["c_mass"], mc["c_lap"], mc["detj"])
            if mc["bc"] != "periodic":
                h.set_dirichlet(np.zeros(mesh.nV))
            rhs = _dev(_host_inputs(mc, seed * 1024 + i)["rhs"])
            f = torch.zeros(mesh.n, dtype=torch.float64, device="cuda")
            torch.cuda.synchronize()
            se_amd.check(lib.se_helm_rhs_dev(h.h, rhs.data_ptr(), f.data_ptr()), "se_helm_rhs_dev")
            ctx.synchronize()
            st["helms"].append(h)
            st["f"].append(f)
            st["xp"].append(st["out"][where[i][0]].data_ptr() + 8 * where[i][1])
        st["batch"] = se_amd.Batch(ctx, st["helms"])
        st["fp"] = [t.data_ptr() for t in st["f"]]
    else:
        mesh = st["mesh"] = _mesh(ctx, case)
        d = _host_inputs(case, seed)
        if case["kind"] in ("solve", "apply"):
            h = st["helm"] = se_amd.Helm(mesh, case["c_mass"], case["c_lap"], case["detj"])
            st["sol"] = _dev(d["wall"])
            if case["bc"] != "periodic":
                h.set_dirichlet(d["wall"].ravel())
            if case["kind"] == "solve":
                st["rhs"] = _dev(d["rhs"])
            else:
                st["x"] = _dev(d["x"])
                st["y"] = torch.zeros_like(st["x"])
        elif case["kind"] == "advect":
            st["dt"] = d["dt"]
            for k in ("psi", "psip", "q", "qp"):
                st[k] = _dev(d[k])
            st["vel"] = torch.zeros(2 * mesh.nV, dtype=torch.float64, device="cuda")
            st["velp"] = torch.zeros_like(st["vel"])
            st["out"] = torch.zeros_like(st["q"])
            st["dep"] = torch.zeros(mesh.nV, dtype=torch.int32, device="cuda")
        else:
            qg = st["qg"] = se_amd.QG(mesh, 100.0, 1.0)
            if case["drag"]:
                qg.set_dissipation(0.0, case["drag"])
            st["psi"], st["om"], st["dt"] = d["psi"][0].ravel(), d["om"][0].ravel(), d["dt"]
    torch.cuda.synchronize()
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "stream":
        srv = st["server"]
        ids = [srv.submit(req, *fields, dt=dt) for req, fields, dt in st["reqs"]]
        return [torch.from_numpy(f) for i in ids for f in srv.wait(i)[1]]
    if kind == "solve":
        prec, pc = SOLVERS[case["solver"]]
        st["helm"].solve_dev(st["rhs"].data_ptr(), st["sol"].data_ptr(), precision=prec, preconditioner=pc,
                             null_space=case["null"])
        return st["sol"]
    if kind == "batch":
        prec, pc = SOLVERS[case["solver"]]
        st["batch"].pcg_dev(st["fp"], st["xp"], precision=prec, preconditioner=pc)
        return st["out"]
    if kind == "apply":
        st["helm"].apply_dev(st["x"].data_ptr(), st["y"].data_ptr())
        return st["y"]
    if kind == "advect":
        lib, m = se_amd.lib(), st["mesh"].h
        p = {k: st[k].data_ptr() for k in ("psi", "psip", "q", "qp", "vel", "velp", "out", "dep")}
        se_amd.check(lib.se_genvel_dev(m, p["psi"], p["vel"]), "se_genvel_dev")
        if case["order"] == 1:
            se_amd.check(lib.se_sl_advect_dev(m, p["q"], case["dofs"], p["vel"], st["dt"], p["out"], p["dep"]),
                         "se_sl_advect_dev")
            return [st["vel"], st["out"], st["dep"]]
        se_amd.check(lib.se_genvel_dev(m, p["psip"], p["velp"]), "se_genvel_dev")
        se_amd.check(lib.se_sl_advect2_dev(m, p["q"], p["qp"], case["dofs"], p["vel"], p["velp"], st["dt"], p["out"]),
                     "se_sl_advect2_dev")
        return [st["vel"], st["velp"], st["out"]]
    prec, pc = SOLVERS[case["solver"]]
    st["qg"].set_state(st["psi"], st["om"])
    for _ in range(case["steps"]):
        st["qg"].step(st["dt"], precision=prec, preconditioner=pc)
    return [torch.from_numpy(f) for f in st["qg"].state()]


# ---------------------------------------------------------------------------
# work


def _apply_flops(c):
    return c["ex"] * c["ey"] * (8.0 * (c["p"] + 1) ** 3 + 4.0 * (c["p"] + 1) ** 2)


def _sl_flops(c):
    # per node: one set of 1-D cardinal functions and a tensor sum per interpolation
    return (c["ex"] * c["p"] + 1) * (c["ey"] * c["p"] + 1) * (4.0 * (c["p"] + 1) ** 2 + 12.0 * (c["p"] + 1))


def work(case):
    """Inputs read once, outputs written once; the flops of one operator product per solve
    (a direct inverse of a separable operator needs no more of that order), of the
    interpolations of an advection, and their sum over the steps of a model."""
    kind = case["kind"]
    if kind == "stream":
        ws = [(_nodes(r), r) for r in _requests(case)]
        return {"bytes": sum(8.0 * 8.0 * n for n, _ in ws),
                "flops": sum(r["steps"] * (2.0 * 4.0 * _sl_flops(r) + 2.0 * _apply_flops(r)) for _, r in ws)}
    if kind == "batch":
        ms = _members(case)
        return {"bytes": sum(16.0 * math.prod(_free_shape(m)) for m in ms), "flops": sum(_apply_flops(m) for m in ms)}
    n = _nodes(case)
    if kind in ("solve", "apply"):
        return {"bytes": 16.0 * n, "flops": _apply_flops(case)}
    if kind == "advect":
        if case["order"] == 1:
            return {"bytes": n * (8.0 + 16.0 + 16.0 * case["dofs"] + 4.0), "flops": 2.0 * _sl_flops(case)}
        return {"bytes": n * (2 * 8.0 + 2 * 16.0 + 24.0 * case["dofs"]), "flops": 4.0 * _sl_flops(case)}
    per = 3.0 * _sl_flops(case) + (2.0 if case["drag"] else 1.0) * _apply_flops(case)
    return {"bytes": 32.0 * n, "flops": case["steps"] * per}


# ---------------------------------------------------------------------------
# the same outputs in plain numpy


def _nodes(c):
    return (c["ex"] * c["p"] + 1) * (c["ey"] * c["p"] + 1)


def _free(ne, p, periodic, wall_lo, wall_hi):
    """First and past-the-last unfolded node of the unknowns of one direction."""
    return (1 if wall_lo else 0), ne * p + (0 if periodic or wall_hi else 1)


def _free_ranges(c):
    per, (b, t, l, r) = BCS[c.get("bc", "channel")]
    return _free(c["ex"], c["p"], per[0], l, r), _free(c["ey"], c["p"], per[1], b, t)


def _free_shape(c):
    (x0, x1), (y0, y1) = _free_ranges(c)
    return y1 - y0, x1 - x0


def _wall_mask(c):
    _, (b, t, l, r) = BCS[c["bc"]]
    m = np.zeros((c["ey"] * c["p"] + 1, c["ex"] * c["p"] + 1), dtype=bool)
    m[0, :] |= bool(b)
    m[-1, :] |= bool(t)
    m[:, 0] |= bool(l)
    m[:, -1] |= bool(r)
    return m


def _line_ops(ne, p, L):
    """Unfolded mass weights and stiffness of one direction."""
    _, w, D = gll(p)
    h = L / ne / 2.0
    G = D.T @ (w[:, None] * D) / h
    n = ne * p + 1
    m, K = np.zeros(n), np.zeros((n, n))
    for e in range(ne):
        s = slice(e * p, e * p + p + 1)
        m[s] += h * w
        K[s, s] += G
    return m, K, h


def _fold(v, periodic, axis):
    """Adds the last line of a periodic direction to the first."""
    if not periodic:
        return v
    v = np.moveaxis(np.array(v), axis, 0)
    v[0] += v[-1]
    return np.moveaxis(v[:-1], 0, axis)


class _Separable:
    """cm M + cl K of a case, restricted to its unknowns."""

    eig = {}

    def __init__(self, c):
        self.c = c
        L = _domain(c)
        self.per = BCS[c.get("bc", "channel")][0]
        self.mx, self.Kx, hx = _line_ops(c["ex"], c["p"], L)
        self.my, self.Ky, hy = _line_ops(c["ey"], c["p"], L)
        self.cm, self.cl = c["c_mass"], c["c_lap"] / (1.0 if c["detj"] else hx * hy)
        (self.x0, self.x1), (self.y0, self.y1) = _free_ranges(c)

    def full(self, u):
        """The unfolded, unrestricted product."""
        return self.cm * self.my[:, None] * u * self.mx + \
            self.cl * (self.my[:, None] * (u @ self.Kx) + (self.Ky @ u) * self.mx)

    def gather(self, v):
        """Sums of the periodic copies, on the unknowns."""
        v = _fold(_fold(v, self.per[0], 1), self.per[1], 0)
        return v[self.y0:self.y1, self.x0:self.x1]

    def scatter(self, x, field=None):
        """Unknowns to a copy of the field, periodic copies filled."""
        u = np.zeros((len(self.my), len(self.mx))) if field is None else np.array(field)
        u[self.y0:self.y1, self.x0:self.x1] = x
        if self.per[0]:
            u[:, -1] = u[:, 0]
        if self.per[1]:
            u[-1, :] = u[0, :]
        return u

    def apply(self, x):
        return self.gather(self.full(self.scatter(x)))

    def line(self, axis):
        c = self.c
        key = (c["ex"] if axis == 0 else c["ey"], c["p"], _domain(c), self.per[axis],
               (self.x0, self.x1) if axis == 0 else (self.y0, self.y1))
        if key not in self.eig:
            m, K = (self.mx, self.Kx) if axis == 0 else (self.my, self.Ky)
            a, b = (self.x0, self.x1) if axis == 0 else (self.y0, self.y1)
            m = _fold(m, self.per[axis], 0)[a:b]
            K = _fold(_fold(K, self.per[axis], 0), self.per[axis], 1)[a:b, a:b]
            s = 1.0 / np.sqrt(m)
            lam, Q = np.linalg.eigh(s[:, None] * K * s)
            if len(self.eig) > 64:
                self.eig.clear()
            self.eig[key] = (lam, s[:, None] * Q)
        return self.eig[key]

    def inverse(self, f):
        lx, Vx = self.line(0)
        ly, Vy = self.line(1)
        D = self.cm + self.cl * (lx[None, :] + ly[:, None])
        t = Vy.T @ f @ Vx
        null = np.abs(D) < 1e-11 * np.abs(D).max()
        t = np.where(null, 0.0, t / np.where(null, 1.0, D))
        return Vy @ t @ Vx.T

    def solve(self, f, null=False):
        if null:
            f = f - f.mean()
        x = self.inverse(f)
        x = x + self.inverse(f - self.apply(x))
        return x - x.mean() if null else x

    def rhs(self, field):
        return self.gather(self.my[:, None] * field * self.mx)

    def lift(self, wall):
        """Lifting of the wall values of a field."""
        if self.c.get("bc", "channel") == "periodic":
            return 0.0
        return -self.gather(self.full(np.where(_wall_mask({**self.c, "bc": self.c.get("bc", "channel")}), wall, 0.0)))

    def solve_field(self, rhs, sol, null=False, wall=None):
        """A whole Helmholtz solve: M rhs + lifting of `wall` (default: sol's), into sol."""
        return self.scatter(self.solve(self.rhs(rhs) + self.lift(sol if wall is None else wall), null), sol)


def _genvel(c, psi):
    """u = -dpsi/dy, v = dpsi/dx; a vertex between elements takes the lower one."""
    p = c["p"]
    D = gll(p)[2]
    L = _domain(c)

    def deriv(f, ne, axis):
        f = np.moveaxis(f, axis, -1)
        el = np.stack([f[..., e * p:e * p + p + 1] for e in range(ne)], -2) @ D.T * (2.0 * ne / L)
        out = np.empty_like(f)
        out[..., 1:] = el[..., 1:].reshape(f.shape[:-1] + (ne * p,))
        out[..., 0] = el[..., 0, 0]
        return np.moveaxis(out, -1, axis)

    return np.stack([-deriv(psi, c["ey"], 0), deriv(psi, c["ex"], 1)], -1)


def _cfl(c, vel):
    return 0.5 * (_domain(c) / max(c["ex"], c["ey"])) / math.sqrt(np.max(vel[..., 0] ** 2 + vel[..., 1] ** 2))


def _cardinals(p, s):
    """Cardinal functions at local coordinates s, by products: (len(s), p + 1)."""
    x = gll(p)[0]
    out = np.ones((len(s), p + 1))
    for j in range(p + 1):
        for k in range(p + 1):
            if k != j:
                out[:, j] *= (s - x[k]) / (x[j] - x[k])
    return out


def _interp(c, fields, pt):
    """Fields [nV1][nV0][d] at points (k, 2)."""
    p, L = c["p"], _domain(c)
    loc = []
    for d, ne in ((0, c["ex"]), (1, c["ey"])):
        dx = L / ne
        e = np.clip(np.floor(pt[:, d] / dx).astype(int), 0, ne - 1)
        loc.append((e * p, _cardinals(p, np.clip((pt[:, d] - e * dx) * (2.0 / dx) - 1.0, -1.0, 1.0))))
    (ix, wx), (iy, wy) = loc
    outs = []
    for f in fields:
        acc = np.zeros((len(pt), f.shape[-1]))
        for j in range(p + 1):
            row = np.zeros_like(acc)
            for i in range(p + 1):
                row += wx[:, i:i + 1] * f[iy + j, ix + i]
            acc += wy[:, j:j + 1] * row
        outs.append(acc)
    return outs


def _wrap(c, pt):
    per = BCS[c.get("bc", "channel")][0]
    L = _domain(c)
    for d in range(2):
        if per[d]:
            pt[:, d] = np.where(pt[:, d] < 0.0, L + pt[:, d], np.where(pt[:, d] > L, pt[:, d] - L, pt[:, d]))
        else:
            pt[:, d] = np.clip(pt[:, d], 0.0, L)
    return pt


def _advect(c, q, qp, vel, velp, dt):
    """Semi-Lagrangian step of q [nV1][nV0][d]: first order (velp None) or second order."""
    L = _domain(c)
    X, Y = _line(c["ex"], c["p"], 0.0, L), _line(c["ey"], c["p"], 0.0, L)
    o = np.stack([a.ravel() for a in np.meshgrid(X, Y)], 1)

    def back(pt, v0, vh):
        xh = _wrap(c, pt - 0.5 * dt * v0)
        return _wrap(c, pt - dt * _interp(c, [vh], xh)[0])

    if velp is None:
        out = _interp(c, [q], back(o, vel.reshape(-1, 2), vel))[0]
    else:
        x1 = back(o, (2.0 * vel - velp).reshape(-1, 2), 1.5 * vel - 0.5 * velp)
        q1, v1 = _interp(c, [q, vel], x1)
        x2 = back(x1, v1, 0.5 * vel + 0.5 * velp)
        out = 2.0 * q1 - 0.5 * _interp(c, [qp], x2)[0]
    out = out.reshape(q.shape)
    return _copies(c, out)


def _copies(c, f):
    per = BCS[c.get("bc", "channel")][0]
    if per[0]:
        f[:, -1] = f[:, 0]
    if per[1]:
        f[-1, :] = f[0, :]
    return f


def _relax(c, alpha, qhat, a):
    """The advected PV over a, averaged over periodic copies; wall rows keep alpha."""
    out = np.array(alpha)
    m = qhat / a
    m[:, 0] = 0.5 * (m[:, 0] + m[:, -1])
    out[1:-1, :-1] = m[1:-1, :-1]
    out[:, -1] = out[:, 0]
    return out


def _qg_exact(c, d):
    """Steps of the one-layer channel model with linear drag."""
    F, beta, r, dt = 100.0, 1.0, c["drag"], d["dt"]
    Y = _line(c["ey"], c["p"], 0.0, 1.0)[:, None]
    psi, om = d["psi"][0], d["om"][0]
    prev = None
    A = _Separable({**c, "c_mass": -F, "c_lap": -1.0, "detj": 0})
    for _ in range(c["steps"]):
        alpha = om - F * psi + beta * Y
        vel = _genvel(c, psi)
        if prev is None:
            a = 1.0
            qh = _advect(c, alpha[..., None], None, vel, None, dt)[..., 0]
        else:
            a = 1.5
            ap = prev[1] - F * prev[0] + beta * Y
            qh = _advect(c, alpha[..., None], ap[..., None], vel, _genvel(c, prev[0]), dt)[..., 0]
        q = qh
        if r:
            ph = np.zeros_like(psi)
            if a != 1.0:
                ph[[0, -1]] = 1.5 * psi[[0, -1]]
            ph = A.solve_field(qh - a * beta * Y, ph, wall=np.zeros_like(psi))
            q = qh - dt * r * (qh + F * ph - a * beta * Y)
        prev = (psi, om)
        al = _relax(c, alpha, q, a)
        psi = A.solve_field(al - beta * Y, psi)
        om = al + F * psi - beta * Y
    return psi, om


def _qg2_exact(c, d):
    """Steps of the two-layer model; the first step relaxes layer 1 only."""
    F, beta, dt = 200.0, 1.0, d["dt"]
    Y = _line(c["ey"], c["p"], 0.0, 1.0)[:, None]
    psi, om = list(d["psi"]), list(d["om"])
    prev = None
    H = _Separable({**c, "c_mass": -2.0 * F, "c_lap": -1.0, "detj": 0})
    P = _Separable({**c, "c_mass": 0.0, "c_lap": -1.0, "detj": 0})
    for _ in range(c["steps"]):
        al = [om[i] + F * (psi[1 - i] - psi[i]) + beta * Y for i in range(2)]
        tau, chi = psi[0] - psi[1], psi[0] + psi[1]
        for i in range(2):
            vel = _genvel(c, psi[i])
            if prev is None:
                if i == 0:
                    al[0] = _relax(c, al[0], _advect(c, al[0][..., None], None, vel, None, dt)[..., 0], 1.0)
            else:
                pp, po = prev
                ap = po[i] + F * (pp[1 - i] - pp[i]) + beta * Y
                qh = _advect(c, al[i][..., None], ap[..., None], vel, _genvel(c, pp[i]), dt)[..., 0]
                al[i] = _relax(c, al[i], qh, 1.5)
        prev = (list(psi), list(om))
        tau = H.solve_field(al[0] - al[1], tau)
        chi = P.solve_field(al[0] + al[1] - 2.0 * beta * Y, chi)
        psi = [0.5 * (tau + chi), 0.5 * (chi - tau)]
        om = [al[i] - F * (psi[1 - i] - psi[i]) - beta * Y for i in range(2)]
    return psi[0], om[0], psi[1], om[1]


def exact(case, seed):
    """What run() returns for these inputs, from the definitions in 64-bit numpy."""
    kind = case["kind"]
    if kind == "stream":
        return [torch.from_numpy(np.ascontiguousarray(f).ravel())
                for i, r in enumerate(_requests(case)) for f in _qg2_exact(r, _host_inputs(r, seed * 64 + i))]
    if kind == "batch":
        members = _members(case)
        where, sizes = _layout(members)
        out = [torch.zeros(n, dtype=torch.float64) for n in sizes]
        for i, (mc, (k, o)) in enumerate(zip(members, where)):
            A = _Separable(mc)
            x = A.solve(A.rhs(_host_inputs(mc, seed * 1024 + i)["rhs"])).ravel()
            out[k][o:o + x.size] = torch.from_numpy(x)
        return out
    d = _host_inputs(case, seed)
    if kind == "solve":
        u = _Separable(case).solve_field(d["rhs"], d["wall"], case["null"])
        return torch.from_numpy(np.ascontiguousarray(u).ravel())
    if kind == "apply":
        A = _Separable(case)
        return torch.from_numpy(np.ascontiguousarray(A.apply(d["x"].reshape(_free_shape(case)))).ravel())
    if kind == "advect":
        vel, velp = _genvel(case, d["psi"]), _genvel(case, d["psip"])
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a).ravel())
        if case["order"] == 1:
            # departure elements are whole numbers decided at round-off: no 64-bit value of their own
            return [t(vel), t(_advect(case, d["q"], None, vel, None, d["dt"])), None]
        return [t(vel), t(velp), t(_advect(case, d["q"], d["qp"], vel, velp, d["dt"]))]
    return [torch.from_numpy(np.ascontiguousarray(f).ravel()) for f in _qg_exact(case, d)]
