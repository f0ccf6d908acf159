"""What a program has this framework do, as cases that can be timed and compared: Burgers runs by
the device driver and by the unmodified task list, ghost exchanges, multigrid solves over
MeshData and on bare arrays, and served solves.

A case is a dict of plain values. `prepare` builds the mesh, the fields and the solver that a
program keeps, with inputs from the seed; `run` is one pass through the public entry points and
returns the fields it updates; `exact` gives the same outputs from plain torch in 64 bits.
"""
import math

import numpy as np
import torch

import parthenon_amd as pa
from parthenon_amd import gmg
from parthenon_amd.burgers import BurgersDriver, DeviceBurgersDriver, make_burgers_mesh

F64 = torch.float64
CFL = 0.4
NG = 4  # ghost cells of the Burgers meshes (WENO5 needs four)


def listed():
    return [
        # A small run, where launches and latency count: 8 blocks, as in the smoke run.
        dict(name="burgers_small", kind="burgers", nx=32, ny=32, nz=32, bx=16, by=16, bz=16,
             scalars=4, recon=0, refine="", cycles=4),
        # The plain Burgers benchmark: 64^3 in 16^3 blocks, 4 scalars, 10 cycles.
        dict(name="burgers_uniform", kind="burgers", nx=64, ny=64, nz=64, bx=16, by=16, bz=16,
             scalars=4, recon=0, refine="", cycles=10),
        # The batched refined step: 64^3 base mesh, a sphere refined two levels, 960 blocks.
        dict(name="burgers_refined", kind="burgers", nx=64, ny=64, nz=64, bx=16, by=16, bz=16,
             scalars=4, recon=0, refine="sphere", cycles=4),
        # The benchmark's larger blocks and its shipped 8 scalars: 128^3 in 32^3 blocks.
        dict(name="burgers_blocks32", kind="burgers", nx=128, ny=128, nz=128, bx=32, by=32,
             bz=32, scalars=8, recon=0, refine="", cycles=2),
        # An adaptive run: every cycle tags and checks the mesh (here it stays as it is).
        dict(name="burgers_adaptive", kind="adaptive", nx=32, ny=32, nz=32, bx=16, by=16, bz=16,
             scalars=4, cycles=4),
        # The unmodified task list (one launch per task) on the refined mesh.
        dict(name="tasks_refined", kind="tasks", nx=64, ny=64, nz=64, bx=16, by=16, bz=16,
             scalars=4, recon=0, refine="sphere", cycles=1),
        # The ghost-exchange microbenchmark: 512 blocks of 16^3, 8 fields, 3 ghosts, in one call.
        dict(name="exchange_fused", kind="exchange", nx=128, ny=128, nz=128, bx=16, by=16, bz=16,
             ng=3, fields=8, ncomp=1, refine="", form="fused"),
        # The same through SendBoundBufs, ReceiveBoundBufs and SetBounds with their buffers.
        dict(name="exchange_tasks", kind="exchange", nx=128, ny=128, nz=128, bx=16, by=16, bz=16,
             ng=3, fields=8, ncomp=1, refine="", form="tasks"),
        # The mixed-precision Poisson solve: 256^3 in 32^3 blocks to 1e-10.
        dict(name="poisson_mixed", kind="poisson", n=256, block=32, precision="mixed"),
        # A small solve on a bare array in FP64, where levels are launch bound.
        dict(name="poisson_array", kind="array", n=64, precision="fp64"),
        # A solve on a refined mesh: 128^3 in 16^3 blocks, the centre refined one level.
        dict(name="poisson_refined", kind="leaf", ndim=3, nb=8, block=16, level=1, lo=3, hi=4),
        # Served solves: ten requests of the served sizes in their proportions, all waiting.
        dict(name="poisson_served", kind="served", n32=4, n64=3, n128=2, n192=1, n48=0, n96=0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mesh(rng, most, cubic):
    """Mesh and block sizes: blocks of 8 to 32 cells, odd multiples among them, at most `most`
    cells."""
    while True:
        if cubic or rng.random() < 0.6:
            b = [rng.choice((8, 16, 16, 16, 32))] * 3
        else:
            b = [rng.choice((8, 10, 12, 16, 20, 24, 32)) for _ in range(3)]
        nb = [rng.randint(1, 8) for _ in range(3)]
        n = [b[d] * nb[d] for d in range(3)]
        target = _log(rng, 4096, most)
        if n[0] * n[1] * n[2] <= target and n[0] * n[1] * n[2] * 8 >= target:
            return dict(nx=n[0], ny=n[1], nz=n[2], bx=b[0], by=b[1], bz=b[2])


def draw(rng):
    kind = rng.choice(("burgers", "burgers", "adaptive", "tasks", "exchange", "exchange",
                       "poisson", "array", "leaf", "leaf", "served"))
    if kind in ("burgers", "tasks"):
        refine = rng.choice(("", "", "sphere", "box"))
        if refine:  # even block sizes, at least 4 blocks a side; the refined part stays small
            b = rng.choice((8, 16, 16))
            n = b * rng.randint(3, 4 if refine == "sphere" else 5)
            c = dict(nx=n, ny=n, nz=n, bx=b, by=b, bz=b)
        else:
            c = _mesh(rng, 96 ** 3, False)
        return dict(kind=kind, **c, scalars=rng.randint(1, 10), recon=rng.choice((0, 0, 0, 1)),
                    refine=refine, cycles=1 if kind == "tasks" else rng.randint(1, 4))
    if kind == "adaptive":
        b = rng.choice((8, 16))
        return dict(kind=kind, nx=b * 2, ny=b * 2, nz=b * rng.choice((2, 4)), bx=b, by=b, bz=b,
                    scalars=rng.randint(1, 8), cycles=rng.randint(1, 4))
    if kind == "exchange":
        refine = rng.choice(("", "", "box"))
        if refine:
            b = rng.choice((8, 16))
            n = b * rng.randint(3, 6)
            c = dict(nx=n, ny=n, nz=n, bx=b, by=b, bz=b)
            ng = rng.choice((2, 4))
        else:
            c = _mesh(rng, 128 ** 3, False)
            ng = rng.choice((2, 3, 4))
        return dict(kind=kind, **c, ng=ng, fields=rng.randint(1, 8), ncomp=rng.choice((1, 1, 3)),
                    refine=refine, form=rng.choice(("fused", "tasks")))
    if kind == "poisson":
        n = 16 * rng.choice((1, 2, 3, 4, 6, 8, 12, 16))
        return dict(kind=kind, n=n, block=rng.choice([b for b in (16, 32) if n % b == 0]),
                    precision=rng.choice(("mixed", "fp64")))
    if kind == "array":
        return dict(kind=kind, n=rng.choice((16, 24, 32, 40, 48, 56, 64, 80, 96, 112, 128)),
                    precision=rng.choice(("mixed", "fp64")))
    if kind == "leaf":
        ndim = rng.choice((2, 3))
        nb = rng.choice((2, 4, 6, 8, 12) if ndim == 2 else (2, 3, 4, 6, 8))
        lo = rng.randint(0, nb - 1)
        return dict(kind=kind, ndim=ndim, nb=nb, block=rng.choice((8, 16, 32) if ndim == 2 else
                                                                  (8, 16) if nb < 8 else (8,)),
                    level=rng.choice((0, 1, 1)), lo=lo, hi=min(nb - 1, lo + rng.randint(0, 1)))
    return dict(kind="served", n32=rng.randint(1, 8), n64=rng.randint(0, 4),
                n128=rng.randint(0, 2), n192=0, n48=rng.randint(0, 4), n96=rng.randint(0, 2))


# ---- what the cases share -------------------------------------------------------------------
class _Device:
    """Device memory of a field for torch (the pointers that a program hands its own kernels)."""

    def __init__(self, pointer, shape):
        self.__cuda_array_interface__ = dict(data=(pointer, False), shape=tuple(shape),
                                             typestr="<f8", version=3)


def _field(md, name):
    return torch.as_tensor(_Device(md.pointers(name)[0], md.mesh.field_shape(name)),
                           device="cuda")


def _interior(a, ng):
    sl = [slice(g, a.shape[-1 - d] - g) for d, g in enumerate(ng)]
    return a[..., sl[2], sl[1], sl[0]]


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _centres(mesh):
    """Cell centres of the interiors of a mesh's blocks: three arrays [block, 1, k, j, i]."""
    blocks = [mesh.block(q) for q in range(mesh.nblocks)]
    lo = torch.tensor([b["xmin"] for b in blocks], dtype=F64, device="cuda")
    hi = torch.tensor([b["xmax"] for b in blocks], dtype=F64, device="cuda")
    out = []
    for d in range(3):
        c = torch.arange(mesh.n[d], dtype=F64, device="cuda") + 0.5
        x = lo[:, d, None] + c[None] * ((hi[:, d] - lo[:, d]) / mesh.n[d])[:, None]
        shape = [mesh.nblocks, 1, 1, 1, 1]
        shape[4 - d] = mesh.n[d]
        out.append(x.reshape(shape))
    return out


def _root(nb, ndim):
    """Levels that the forest of a block grid has above it: halvings of every dimension."""
    if ndim < 3:
        return 0
    r = 0
    while all(v % (2 << r) == 0 for v in nb):
        r += 1
    return r


def _order(nb, ndim):
    """Positions (x, y, z) of a uniform grid's blocks in block order, the Morton order of their
    positions."""
    def morton(p):
        return sum(((p[d] >> bit) & 1) << (3 * bit + d) for bit in range(12) for d in range(3))
    return sorted(((x, y, z) for z in range(nb[2]) for y in range(nb[1]) for x in range(nb[0])),
                  key=morton)


def _bricks(padded, nb, n, ng, ndim):
    """Blocks with ghosts [block, comp, k, j, i] of an array [comp, z, y, x] with ghosts."""
    return torch.stack([padded[:, z * n[2]:(z + 1) * n[2] + 2 * ng[2],
                               y * n[1]:(y + 1) * n[1] + 2 * ng[1],
                               x * n[0]:(x + 1) * n[0] + 2 * ng[0]]
                        for x, y, z in _order(nb, ndim)])


def _global(bricks, nb, n, ndim):
    """The array [comp, z, y, x] of blocks without ghosts."""
    out = torch.empty(bricks.shape[1], nb[2] * n[2], nb[1] * n[1], nb[0] * n[0], dtype=F64,
                      device=bricks.device)
    for q, (x, y, z) in enumerate(_order(nb, ndim)):
        out[:, z * n[2]:(z + 1) * n[2], y * n[1]:(y + 1) * n[1], x * n[0]:(x + 1) * n[0]] = \
            bricks[q]
    return out


def _wrap(a, ng):
    for d in range(3):
        g = ng[d]
        if g:
            n = a.shape[-1 - d]
            idx = (torch.arange(-g, n + g, device=a.device)) % n
            a = a.index_select(a.dim() - 1 - d, idx)
    return a


# ---- Burgers ------------------------------------------------------------------------------
def _sizes(c):
    return (c["nx"], c["ny"], c["nz"]), (c["bx"], c["by"], c["bz"])


def _refined(c):
    if c.get("refine") == "sphere":
        return dict(refine_spheres=[((0.0, 0.0, 0.0), 0.25, 2 if c["nx"] >= 4 * c["bx"] else 1)])
    if c.get("refine") == "box":
        return dict(refine_boxes=[((-0.1, 0.1, -0.1, 0.1, -0.1, 0.1), 1)])
    return {}


def _sinusoids(V, seed, x):
    """Sums of four sinusoids per component, seeded amplitudes and phases, at the positions x."""
    r = np.random.default_rng(seed)
    amp, phase = 0.1 + 0.9 * r.random((V, 4)), 2.0 * math.pi * r.random((V, 4))
    out = []
    for v in range(V):
        s = 0.0
        for q in range(4):
            s = s + amp[v, q] * torch.sin(2.0 * math.pi * (q + 1) * x[(v + q) % 3] + phase[v, q])
        out.append(s)
    return out


def _set_sinusoids(mesh, seed):
    md = mesh.mesh_data("base")
    U = _interior(_field(md, "U"), mesh.ng)
    for v, s in enumerate(_sinusoids(U.shape[1], seed, _centres(mesh))):
        U[:, v:v + 1] = s
    torch.cuda.synchronize()


def _prepare_burgers(c, seed):
    nx, block = _sizes(c)
    if c["kind"] == "adaptive":
        # one criterion as in the shipped input, tight enough that every block is refined
        crit = [dict(field="U", comp=3, method="derivative_order_1", refine_tol=1e-6,
                     derefine_tol=0.0)]
        root = _root([nx[d] // block[d] for d in range(3)], 3)
        mesh = make_burgers_mesh(nx, block, NG, c["scalars"],
                                 adaptive=dict(numlevel=root + 1, derefine_count=10,
                                               criteria=crit))
    else:
        mesh = make_burgers_mesh(nx, block, NG, c["scalars"], **_refined(c))
    _set_sinusoids(mesh, seed)
    if c["kind"] == "tasks":
        drv = BurgersDriver(mesh, cfl=CFL, recon=c["recon"])
        drv.initialize(pgen=None)
    else:
        drv = DeviceBurgersDriver(mesh, cfl=CFL, recon=c.get("recon", 0))
        drv.initialize(pgen=None)
    if c["kind"] == "adaptive":
        drv.adaptive_cycles(2)  # the mesh settles: every block refined
    drv.mesh.synchronize()
    return dict(case=c, mesh=mesh, drv=drv, md=mesh.mesh_data("base"))


def _run_burgers(s):
    c, drv = s["case"], s["drv"]
    if c["kind"] == "tasks":
        for _ in range(c["cycles"]):
            drv.cycle()
    elif c["kind"] == "adaptive":
        drv.adaptive_cycles(c["cycles"])
    else:
        drv.cycles(c["cycles"])
    return {"U": _field(s["md"], "U"), "derived": _field(s["md"], "derived")}


def _weno(q):
    """WENO5-Z with its limiter towards linear, of the cell q[2] in q[0] .. q[4]."""
    eps = 10.0 * np.finfo(np.float64).eps
    q0, q1, q2, q3, q4 = q
    t = 13.0 / 3.0
    b0 = t * (q0 - 2 * q1 + q2) ** 2 + (q0 - 4 * q1 + 3 * q2) ** 2 + eps
    b1 = t * (q1 - 2 * q2 + q3) ** 2 + (q3 - q1) ** 2 + eps
    b2 = t * (q2 - 2 * q3 + q4) ** 2 + (q4 - 4 * q3 + 3 * q2) ** 2 + eps
    tau = (b2 - b0).abs()
    z0, z1, z2 = (b0 + tau) / b0, (b1 + tau) / b1, (b2 + tau) / b2

    def side(za, zb, zc, p0, p1, p2, p3, p4):
        w0, w1, w2 = 0.1 * za + eps, 0.6 * zb + eps, 0.3 * zc + eps
        s = 1.0 / (w0 + w1 + w2)
        v = (w0 * (p0 / 3 - 7 * p1 / 6 + 11 * p2 / 6) + w1 * (-p1 / 6 + 5 * p2 / 6 + p3 / 3) +
             w2 * (p2 / 3 + 5 * p3 / 6 - p4 / 6)) * s
        a = 3 * s * w0 * w1 * w2 / (0.3 * w0 * w1 + 0.6 * w0 * w2 + 0.1 * w1 * w2) + eps
        return v, a

    vl, al = side(z0, z1, z2, q0, q1, q2, q3, q4)
    vr, ar = side(z2, z1, z0, q4, q3, q2, q1, q0)
    dq = 0.5 * _mc(q2 - q1, q3 - q2)
    lin = 2 * al * ar / (al + ar)
    return lin * vl + (1 - lin) * (q2 + dq), lin * vr + (1 - lin) * (q2 - dq)


def _mc(dm, dp):
    dc = torch.where(dm * dp > 0, 0.5 * (dm + dp), torch.zeros_like(dm))
    return torch.copysign(torch.minimum(dc.abs(), 2 * torch.minimum(dm.abs(), dp.abs())), dc)


def _rate(U, dx, recon):
    """dU/dt on a periodic uniform grid [comp, z, y, x]."""
    out = torch.zeros_like(U)
    for d in range(3):
        ax = 3 - d

        def at(o, a=U):
            return torch.roll(a, -o, ax)
        if recon == 0:
            ql, qr = _weno([at(-2), at(-1), U, at(1), at(2)])
        else:
            dq = 0.5 * _mc(U - at(-1), at(1) - U)
            ql, qr = U + dq, U - dq
        L, R = torch.roll(ql, 1, ax), qr  # states of each cell's low face
        ul, ur = L[d], R[d]
        zero = torch.zeros_like(ul)
        sl, sr = torch.minimum(torch.minimum(ul, ur), zero), torch.maximum(torch.maximum(ul, ur),
                                                                          zero)
        F = (sr * ul * L - sl * ur * R + sl * sr * (R - L)) / (sr - sl + (sl * sr == 0))
        F[:3] *= 0.5
        out -= (torch.roll(F, -1, ax) - F) / dx[d]
    return out


def _exact_burgers(c, seed):
    if c["kind"] == "adaptive" or c.get("refine"):
        return None
    nx, block = _sizes(c)
    dx = [1.0 / n for n in nx]
    x = []
    for d in range(3):
        shape = [1, 1, 1]
        shape[2 - d] = nx[d]
        x.append((-0.5 + (torch.arange(nx[d], dtype=F64, device="cuda") + 0.5) * dx[d]).reshape(
            shape))
    U = torch.stack([s.expand(nx[2], nx[1], nx[0])
                     for s in _sinusoids(3 + c["scalars"], seed, x)]).contiguous()

    def estimate(U):
        return CFL * float((1.0 / sum(U[d].abs() / dx[d] for d in range(3))).min())
    dt = estimate(U)
    for _ in range(c["cycles"]):
        one = U + dt * _rate(U, dx, c["recon"])
        U = 0.5 * one + 0.5 * U + 0.5 * dt * _rate(one, dx, c["recon"])
        dt = min(2.0 * dt, estimate(U))
    nb = [nx[d] // block[d] for d in range(3)]
    g = (NG, NG, NG)
    derived = 0.5 * U[3] * (U[0] ** 2 + U[1] ** 2 + U[2] ** 2)
    inner = _bricks(derived[None], nb, block, (0, 0, 0), 3)
    return {"U": _bricks(_wrap(U, g), nb, block, g, 3),
            "derived": torch.nn.functional.pad(inner, (NG,) * 6)}


# ---- exchange -------------------------------------------------------------------------------
def _exchange_inputs(c, seed, shape):
    g = _generator(seed)
    return [2.0 * torch.rand(shape, generator=g, dtype=F64, device="cuda") - 1.0
            for _ in range(c["fields"])]


def _prepare_exchange(c, seed):
    nx, block = _sizes(c)
    m = pa.Mesh(nx, block, c["ng"], **_refined(c))
    for f in range(c["fields"]):
        m.add_field("q%d" % f, c["ncomp"])
    m.finalize()
    md = m.mesh_data("base")
    shape = (m.nblocks, c["ncomp"], m.n[2], m.n[1], m.n[0])
    for f, v in enumerate(_exchange_inputs(c, seed, shape)):
        _interior(_field(md, "q%d" % f), m.ng).copy_(v)
    torch.cuda.synchronize()
    return dict(case=c, mesh=m, md=md)


def _run_exchange(s):
    if s["case"]["form"] == "fused":
        pa.exchange_fused(s["md"])
    else:
        pa.exchange(s["md"])
    return {"q%d" % f: _field(s["md"], "q%d" % f) for f in range(s["case"]["fields"])}


def _exact_exchange(c, seed):
    if c["refine"]:
        return None
    nx, block = _sizes(c)
    nb = [nx[d] // block[d] for d in range(3)]
    g = (c["ng"],) * 3
    shape = (nb[0] * nb[1] * nb[2], c["ncomp"], block[2], block[1], block[0])
    return {"q%d" % f: _bricks(_wrap(_global(v, nb, block, 3), g), nb, block, g, 3)
            for f, v in enumerate(_exchange_inputs(c, seed, shape))}


# ---- Poisson ----------------------------------------------------------------------------------
REL = 1e-10  # every solve runs until its residual is this small beside the right-hand side


def _blobs(seed, x, lo, hi):
    """16 Gaussian blobs of either sign at seeded places of [lo, hi]^3."""
    r = np.random.default_rng(seed)
    out = 0.0
    for _ in range(16):
        c = lo + (hi - lo) * r.uniform(0.1, 0.9, 3)
        w = (hi - lo) * r.uniform(0.02, 0.08)
        a = r.choice([-1.0, 1.0])
        out = out + a * torch.exp(-sum((x[d] - c[d]) ** 2 for d in range(3)) / (w * w))
    return out


def _axes(n):
    out = []
    for d in range(3):
        shape = [1, 1, 1]
        shape[2 - d] = n
        out.append(((torch.arange(n, dtype=F64, device="cuda") + 0.5) / n).reshape(shape))
    return out


def _solve_exactly(b):
    """u of the 7-point problem (u = 0 on the faces of the unit cube) by the sines that
    diagonalise it."""
    n = b.shape[-1]
    i = torch.arange(n, dtype=F64, device=b.device)
    S = torch.sin(math.pi * (i[:, None] + 1.0) * (i[None] + 0.5) / n)  # [mode, cell]
    S = S / S.norm(dim=1, keepdim=True)
    lam = -(2.0 - 2.0 * torch.cos(math.pi * (i + 1.0) / n)) * n * n

    def along(M, a):
        for _ in range(3):  # the last axis each time, then the axes rotate
            a = (a.reshape(-1, n) @ M.T.contiguous()).reshape(n, n, n).permute(2, 0, 1)
            a = a.contiguous()
        return a
    t = along(S, b)
    t = t / (lam[:, None, None] + lam[None, :, None] + lam[None, None, :])
    return along(S.T.contiguous(), t)


def _prepare_poisson(c, seed):
    n, b = c["n"], c["block"]
    m = pa.Mesh((n,) * 3, (b,) * 3, 2, xmin=(0.0,) * 3, xmax=(1.0,) * 3, periodic=(0, 0, 0),
                bcs=("fixed_face",) * 6)
    m.add_field("u", 1)
    m.add_field("rhs", 1)
    m.finalize()
    md = m.mesh_data("base")
    rhs = _blobs(seed, _centres(m), 0.0, 1.0)
    _interior(_field(md, "rhs"), m.ng).copy_(rhs)
    torch.cuda.synchronize()
    tol = REL * float(rhs.square().mean().sqrt())
    solver = gmg.MeshMGSolver(m, "u", "rhs", gmg.MeshMGParams(
        max_iters=100, residual_tolerance=tol, precision=c["precision"]))
    return dict(case=c, mesh=m, md=md, solver=solver)


def _run_mesh_solve(s):
    md = s["md"]
    gmg.set_to_zero(md, "u")
    s["solver"].setup(md)
    s["solver"].solve(md)
    u = _field(md, "u")
    if s["case"]["kind"] == "poisson":
        return {"u": u}
    return {"u": u, "solution": _interior(u, s["mesh"].ng)}


def _exact_poisson(c, seed):
    n, b, g = c["n"], c["block"], 2
    u = _solve_exactly(_blobs(seed, _axes(n), 0.0, 1.0))
    for d in range(3):  # ghosts of a face at 0: the mirrored cell, negated
        ax = 2 - d
        u = torch.cat([-u.narrow(ax, 0, g).flip(ax), u, -u.narrow(ax, n - g, g).flip(ax)], ax)
    return {"u": _bricks(u[None], (n // b,) * 3, (b,) * 3, (g,) * 3, 3)}


def _prepare_array(c, seed):
    s = gmg.MGSolver(c["n"], c["precision"], gmg.MGParams(residual_tolerance=REL))
    s.set_rhs(_blobs(seed, _axes(c["n"]), 0.0, 1.0).cpu().numpy())
    return dict(case=c, solver=s)


def _run_array(s):
    s["solver"].reset()
    s["solver"].solve()
    return {"u": s["solver"].solution()}


def _exact_array(c, seed):
    return {"u": _solve_exactly(_blobs(seed, _axes(c["n"]), 0.0, 1.0))}


def _leaf_shape(c):
    d3 = c["ndim"] == 3
    n = c["nb"] * c["block"]
    return (n, n, n if d3 else 1), (c["block"], c["block"], c["block"] if d3 else 1)


def _leaves(c):
    """(level, position) of the blocks of a refined mesh in block order."""
    nb = (c["nb"], c["nb"], c["nb"] if c["ndim"] == 3 else 1)
    out = []
    for p in _order(nb, c["ndim"]):
        if c["level"] and all(c["lo"] <= p[d] <= c["hi"] for d in range(c["ndim"])):
            for m in range(1 << c["ndim"]):
                out.append((1, tuple(2 * p[d] + ((m >> d) & 1) if d < c["ndim"] else 0
                                     for d in range(3))))
        else:
            out.append((0, p))
    return out


def _smooth(seed, ndim, x):
    """A seeded field that vanishes on the faces of [-1, 1]^ndim."""
    r = np.random.default_rng(seed)
    out = 0.0
    for _ in range(12):
        v = r.normal()
        for d in range(ndim):
            v = v * torch.sin(math.pi * r.integers(1, 9) * 0.5 * (x[d] + 1.0))
        out = out + v
    return out


def _prepare_leaf(c, seed):
    nx, block = _leaf_shape(c)
    nd = c["ndim"]
    boxes = []
    if c["level"]:
        w = 2.0 / c["nb"]
        box = []
        for d in range(3):
            box += [-1.0 + w * (c["lo"] + 0.25), -1.0 + w * (c["hi"] + 0.75)] if d < nd else [0.0,
                                                                                              1.0]
        boxes = [(tuple(box), c["level"])]
    m = pa.Mesh(nx, block, 2, xmin=tuple(-1.0 if d < nd else 0.0 for d in range(3)),
                xmax=(1.0,) * 3, periodic=tuple(int(d >= nd) for d in range(3)),
                bcs=tuple("fixed_face" if d < nd else "periodic" for d in range(3)
                          for _ in range(2)), refine_boxes=boxes)
    m.add_field("u", 1)
    m.register_refinement_ops("u", "linear")
    m.add_field("rhs", 1)
    m.finalize()
    md = m.mesh_data("base")
    # the right-hand side of a known solution, as the poisson_gmg package's use_exact_rhs
    _interior(_field(md, "u"), m.ng).copy_(_smooth(seed, nd, _centres(m)))
    torch.cuda.synchronize()
    pa.exchange_fused(md)
    gmg.PoissonEquation().Ax(md, "u", "rhs")
    m.synchronize()
    rhs = _interior(_field(md, "rhs"), m.ng)
    tol = REL * float(rhs.square().mean().sqrt())
    solver = gmg.MeshMGSolver(m, "u", "rhs", gmg.MeshMGParams(
        max_iters=60, residual_tolerance=tol, precision="fp64", smoother="SRJ2"))
    return dict(case=c, mesh=m, md=md, solver=solver)


def _exact_leaf(c, seed):
    _, n = _leaf_shape(c)
    leaves = _leaves(c)
    x = []
    for d in range(3):
        cells = torch.arange(n[d], dtype=F64, device="cuda") + 0.5
        h = torch.tensor([2.0 / c["nb"] / (1 << lev) for lev, _ in leaves], dtype=F64,
                         device="cuda")
        at = torch.tensor([p[d] for _, p in leaves], dtype=F64, device="cuda")
        shape = [len(leaves), 1, 1, 1, 1]
        shape[4 - d] = n[d]
        x.append((-1.0 + h[:, None] * (at[:, None] + cells[None] / n[d])).reshape(shape))
    u = _smooth(seed, c["ndim"], x)
    return {"u": None, "solution": u.expand(len(leaves), 1, n[2], n[1], n[0]).contiguous()}


def _requests(c):
    return [n for n in (32, 48, 64, 96, 128, 192) for _ in range(c["n%d" % n])]


def _prepare_served(c, seed):
    # a run solves every submitted request again, so the limit on V-cycles counts all runs
    server = gmg.Server("mixed", gmg.MGParams(residual_tolerance=REL, max_iters=10 ** 8),
                        keep_solutions=True)
    ids = [server.submit(n, seed * 100 + q) for q, n in enumerate(_requests(c))]
    server.run(realtime=False)  # the server's memory pool is warm, as in service
    return dict(case=c, server=server, ids=ids)


def _run_served(s):
    s["server"].run(realtime=False)
    return [s["server"].solution(q) for q in s["ids"]]


def _served_rhs(n, seed):
    """The blob field that a request's seed stands for."""
    state, mask = seed, (1 << 64) - 1

    def uniform():
        nonlocal state
        state = (state + 0x9E3779B97F4A7C15) & mask
        z = state
        z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & mask
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
        return ((z ^ (z >> 31)) >> 11) * 2.0 ** -53
    x = _axes(n)
    out = 0.0
    for _ in range(16):
        c = [0.1 + 0.8 * uniform() for _ in range(3)]
        w = 0.02 + 0.06 * uniform()
        a = -1.0 if uniform() < 0.5 else 1.0
        out = out + a * torch.exp(-sum((x[d] - c[d]) ** 2 for d in range(3)) / (w * w))
    return out


def _exact_served(c, seed):
    return [_solve_exactly(_served_rhs(n, seed * 100 + q)) for q, n in enumerate(_requests(c))]


_PREPARE = dict(burgers=_prepare_burgers, tasks=_prepare_burgers, adaptive=_prepare_burgers,
                exchange=_prepare_exchange, poisson=_prepare_poisson, array=_prepare_array,
                leaf=_prepare_leaf, served=_prepare_served)
_RUN = dict(burgers=_run_burgers, tasks=_run_burgers, adaptive=_run_burgers,
            exchange=_run_exchange, poisson=_run_mesh_solve, array=_run_array,
            leaf=_run_mesh_solve, served=_run_served)
_EXACT = dict(burgers=_exact_burgers, tasks=_exact_burgers, adaptive=_exact_burgers,
              exchange=_exact_exchange, poisson=_exact_poisson, array=_exact_array,
              leaf=_exact_leaf, served=_exact_served)


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return _RUN[state["case"]["kind"]](state)


def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)


def _cells(c):
    """Interior cells of a case's mesh (refined meshes: from the block counts of the forest)."""
    nx, block = _sizes(c)
    n = nx[0] * nx[1] * nx[2]
    if c["kind"] == "adaptive":
        return 8 * n
    if c.get("refine"):
        m = pa.Mesh(nx, block, NG, **_refined(c))
        m.add_field("q", 1)
        m.plan()
        return m.nblocks * block[0] * block[1] * block[2]
    return n


def _levels(n):
    """Cells of every level of an n^3 hierarchy beside those of the finest."""
    out, m = 0.0, n
    while True:
        out += (m / n) ** 3
        if m % 2 or m == 1:
            return out
        m //= 2


def _solve_work(n, mixed):
    """A multigrid solve to 1e-10: about 22 V-cycles; a V-cycle at the least reads the
    right-hand side and reads and writes the correction on the way down and on the way up, an
    FP64 step reads u, e and b and writes u and r."""
    cells, es = float(n) ** 3, 4 if mixed else 8
    steps = 11 if mixed else 22
    per_cycle, per_step = 5 * es, 3 * 8 + 2 * es
    return dict(bytes=cells * (22 * per_cycle * _levels(n) + steps * per_step),
                flops=cells * (22 * 4 * 12 * _levels(n) + steps * 12))


def work(case):
    c = case
    if c["kind"] in ("burgers", "tasks", "adaptive"):
        # a stage reads its input (the second one the cycle's start too) and writes its output;
        # a reconstruction is about 150 operations for each component and direction
        V, cells = 3 + c["scalars"], _cells(c)
        return dict(bytes=8.0 * c["cycles"] * cells * (5 * V + 1),
                    flops=2.0 * c["cycles"] * cells * V * (3 * 170 + 8))
    if c["kind"] == "exchange":
        # every ghost cell is read once from its owner and written once
        nx, block = _sizes(c)
        blocks = _cells(c) // (block[0] * block[1] * block[2])
        whole = (block[0] + 2 * c["ng"]) * (block[1] + 2 * c["ng"]) * (block[2] + 2 * c["ng"])
        ghosts = whole - block[0] * block[1] * block[2]
        return dict(bytes=16.0 * blocks * ghosts * c["fields"] * c["ncomp"], flops=0.0)
    if c["kind"] == "leaf":
        # 15 V-cycles of two sweeps, a residual and two sweeps over every block
        cells = len(_leaves(c)) * float(c["block"]) ** c["ndim"]
        return dict(bytes=cells * 15 * 8 * 8 * 1.15, flops=cells * 15 * 5 * 14 * 1.15)
    if c["kind"] == "served":
        every = [_solve_work(n, True) for n in _requests(c)]
        return dict(bytes=sum(w["bytes"] for w in every), flops=sum(w["flops"] for w in every))
    return _solve_work(c["n"], c["precision"] == "mixed")


def tolerance(case):
    if case["kind"] == "exchange" and not case["refine"]:
        return "exact"  # copies
    if case["kind"] == "exchange":  # averages and interpolations of at most 8 values
        return {"rel": 1e-15, "max": 1e-14}
    if case["kind"] in ("burgers", "tasks", "adaptive"):
        # runs by two of the driver's stage forms, whose sums have another order, differ by up
        # to 9e-16 (2e-14 at one cell) after three passes
        return {"rel": 1e-14, "max": 5e-13}
    # a solve ends below the residual that it was asked for: solutions are 2e-11 to 5e-10 off
    return {"rel": 2e-9, "max": 8e-8}
