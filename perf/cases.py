"""Workloads whose speed matters to users of pict_amd, through its public entry points.

Every case is one of these programs, over the sizes and options they are run with:

  step    PISO time steps of a `Simulation` (forward): initial state in, velocity and pressure out
  grad    a differentiable rollout with per-step checkpoints and its backward: final velocities, their loss's
          gradients with respect to the initial velocities and the per-cell forcing out
  batch   one step of many independent cavities through `SimulationBatch`
  cg      one pressure system through `SolveLinear` (CG), the mean removed as the driver does
  bicg    one advection system with one right-hand side per velocity component (BiCGStab)
  refine  one pressure system through `SolveLinearRefined` (FP64 accuracy from FP32 correction solves)

Grids are tensor products (uniform or wall-clustered) given as vertex coordinates, periodic or with no-slip walls,
as one block or as two blocks joined along y; `refine` and one kind of `cg` use the numbering of an O-grid of four
blocks.  `exact` restates the discretisation on whole arrays in 64 bits with converged solves; the solver tolerances
of the cases are tight enough that a solve that stops an iteration earlier or later does not show.
"""
import math

import torch

from pict_amd import PISOtorch as P
from pict_amd import PISOtorch_simulation as S
from pict_amd import checkpoint as CK
from pict_amd.batch import SimulationBatch

_DTYPE = {"f32": torch.float32, "f64": torch.float64}


def listed():
    return [
        # the plain lid-driven cavity at its usual 32 x 32: every launch and host call of a step counts
        dict(name="step_cavity_32", kind="step", nx=32, ny=32, nz=0, flow="cavity", blocks=1, steps=2, dtype="f32"),
        # a ragged cavity in double precision, as gradient checks and reference solutions are run
        dict(name="step_cavity_97x61_f64", kind="step", nx=97, ny=61, nz=0, flow="cavity", blocks=1, steps=1,
             dtype="f64"),
        # decaying turbulence on the two-block periodic box: generating training data
        dict(name="step_box_256", kind="step", nx=256, ny=256, nz=0, flow="box", blocks=2, steps=2, dtype="f32"),
        # the same box inside a training loop: rollout, loss, gradients of initial state and forcing
        dict(name="grad_box_256", kind="grad", nx=256, ny=256, nz=0, flow="box", blocks=2, steps=2, dtype="f32"),
        # a training step at a small ragged size
        dict(name="grad_box_75x54", kind="grad", nx=75, ny=54, nz=0, flow="box", blocks=2, steps=2, dtype="f32"),
        # the turbulent channel at its full size, forward
        dict(name="step_channel_192x96x96", kind="step", nx=192, ny=96, nz=96, flow="channel", blocks=1, steps=1,
             dtype="f32"),
        # the channel inside a training loop, full size and a ragged small one
        dict(name="grad_channel_192x96x96", kind="grad", nx=192, ny=96, nz=96, flow="channel", blocks=1, steps=1,
             dtype="f32"),
        dict(name="grad_channel_57x35x30", kind="grad", nx=57, ny=35, nz=30, flow="channel", blocks=1, steps=2,
             dtype="f32"),
        # many small simulations at once: a data set of cavities of mixed sizes and viscosities
        dict(name="batch_64_cavities", kind="batch", count=64, lo=32, hi=256, seed0=0, dtype="f32"),
        # pressure systems on their own: a mid-size 3-D duct, and the O-grid to FP64 accuracy
        dict(name="cg_duct_131x67x45", kind="cg", nx=131, ny=67, nz=45, flow="channel", ogrid=0, dtype="f32"),
        dict(name="refine_ogrid_4x128x128", kind="refine", nx=128, ny=128, nz=0, flow="box", ogrid=1, dtype="f32"),
        # the advection system of a 2-D step on its own, ragged
        dict(name="bicg_box_301x203", kind="bicg", nx=301, ny=203, nz=0, flow="box", ogrid=0, dtype="f32"),
    ]


def draw(rng):
    """One more case: a kind, then sizes spread evenly over the logarithm of their range, odd ones among them."""
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["step", "step", "grad", "grad", "batch", "cg", "cg", "refine", "bicg"])
    if kind == "batch":
        return dict(kind="batch", count=size(8, 48), lo=size(24, 48), hi=size(96, 256), seed0=rng.randrange(1000),
                    dtype="f32")
    if kind == "refine":
        return dict(kind="refine", nx=size(24, 128), ny=size(24, 128), nz=0, flow="box", ogrid=1, dtype="f32")
    three = rng.random() < 0.4
    flow = "channel" if three else rng.choice(["cavity", "box"])
    if three:
        nx, ny, nz = size(24, 192), size(17, 96), size(16, 96)
    else:
        nx, ny, nz = size(24, 320), size(24, 256), 0
    dtype = "f64" if rng.random() < 0.2 else "f32"
    if three and dtype == "f64":  # double precision is for checks, at smaller sizes
        nx, ny, nz = max(nx // 2, 17), max(ny // 2, 16), max(nz // 2, 16)
    if kind in ("cg", "bicg"):
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, flow=flow, ogrid=0, dtype=dtype)
    blocks = 1
    if flow == "box":
        blocks, ny = 2, ny + ny % 2
    steps = 1 if three else rng.choice([1, 2])
    return dict(kind=kind, nx=nx, ny=ny, nz=nz, flow=flow, blocks=blocks, steps=steps, dtype=dtype)


# --------------------------------------------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------------------------------------------

def _cells(case):
    return case["nx"] * case["ny"] * max(case["nz"], 1) * (4 if case.get("ogrid") else 1)


def _axes(case):
    """Vertex positions per axis (x, y[, z]) in 64 bits and whether the axis is periodic."""
    n = [case["nx"], case["ny"]] + ([case["nz"]] if case["nz"] else [])
    lin = lambda lo, hi, k: torch.linspace(lo, hi, k + 1, dtype=torch.float64)  # noqa: E731
    if case["flow"] == "cavity":
        return [lin(0, 1, k) for k in n], [False] * len(n)
    if case["flow"] == "box":
        h = 2 * math.pi / n[0]
        return [lin(0, 2 * math.pi, n[0]), lin(0, n[1] * h, n[1])], [True, True]
    # channel: walls in y with cells clustered towards them, periodic in x and z
    y = torch.tanh(2.0 * lin(-1, 1, n[1])) / math.tanh(2.0)
    return [lin(0, 2 * math.pi, n[0]), y, lin(0, math.pi, n[2])], [True, False, True]


def _flow_parameters(case):
    """(viscosity, lid velocity, largest speed, time step) with the time step at a CFL number of 0.25 to 0.4."""
    x = _axes(case)[0]
    if case["flow"] == "cavity":
        return 0.01, 1.0, 1.0, 0.4 / max(case["nx"], case["ny"])
    if case["flow"] == "box":
        return 1e-3, 0.0, 3.0, 0.25 * float(x[0][1]) / 3.0
    return 1.0 / 180.0, 0.0, 23.55, 0.4 * float(x[0][1]) / 23.55


def _velocity(case, seed):
    """Initial velocity [D, (nz,) ny, nx] in 64 bits: random smooth modes (cavity: a streamfunction that vanishes on
    the walls; box: a k^-5/3-like spectrum; channel: the laminar profile) with Gaussian noise on top."""
    g = torch.Generator().manual_seed(seed)
    verts, _ = _axes(case)
    c = [0.5 * (v[1:] + v[:-1]) for v in verts]
    if case["flow"] == "channel":
        u = torch.randn([3, case["nz"], case["ny"], case["nx"]], generator=g, dtype=torch.float64) * (0.05 * 23.55)
        u[0] += 23.55 * (1.0 - c[1] ** 2)[None, :, None]
        return u
    X, Y = c[0][None, :], c[1][:, None]
    u = torch.zeros([2, case["ny"], case["nx"]], dtype=torch.float64)
    ly = float(verts[1][-1])
    for _ in range(24):
        amp, ph, ps = torch.rand(3, generator=g, dtype=torch.float64).tolist()
        kx, ky = (int(v) for v in torch.randint(1, 9, (2,), generator=g))
        if case["flow"] == "cavity":
            a, b = math.pi * kx, math.pi * ky
            w = (amp - 0.5) * 0.6 / (kx * ky) / math.pi
            u[0] += w * b * torch.sin(a * X) * torch.cos(b * Y)
            u[1] -= w * a * torch.cos(a * X) * torch.sin(b * Y)
        else:
            a, b = float(kx), 2 * math.pi * ky / ly
            w = (amp - 0.5) * 2.0 / (kx ** 2 + ky ** 2) ** (11.0 / 12.0)
            u[0] += w * b * torch.sin(a * X + 6.3 * ph) * torch.cos(b * Y + 6.3 * ps)
            u[1] -= w * a * torch.cos(a * X + 6.3 * ph) * torch.sin(b * Y + 6.3 * ps)
    return u + 0.01 * torch.randn(u.shape, generator=g, dtype=torch.float64)


def _target(case, seed):
    return _velocity(case, seed + 7919)


def _block_slices(case):
    """y ranges of the blocks."""
    k = case["ny"] // case["blocks"]
    return [(i * k, (i + 1) * k) for i in range(case["blocks"])]


def _rounded_axes(case):
    """Vertex positions in the case's precision (what the framework is given), periodic flags."""
    verts, per = _axes(case)
    return [v.to(_DTYPE[case["dtype"]]) for v in verts], per


def _domain(case, seed, name="case"):
    dt = _DTYPE[case["dtype"]]
    verts, per = _rounded_axes(case)
    visc, lid, _, _ = _flow_parameters(case)
    visc = case.get("visc", visc)
    dims = len(verts)
    dom = P.Domain(dims, torch.tensor([visc], dtype=dt), name, dt, "cuda", passiveScalarChannels=0)
    vel = _velocity(case, seed).to(dtype=dt, device="cuda")
    blocks = []
    for lo, hi in _block_slices(case):
        ax = [verts[0], verts[1][lo:hi + 1]] + verts[2:]
        grid = torch.meshgrid(*reversed(ax), indexing="ij")
        b = dom.CreateBlock(vertexCoordinates=torch.stack(list(reversed(grid)))[None].cuda().contiguous(),
                            name="b%d" % lo)
        if not all(per):
            b.CloseAllBoundaries()
        for d, p in enumerate(per):
            if p and not (d == 1 and case["blocks"] > 1):
                b.MakePeriodic("xyz"[d])
        if lid:
            b.CloseBoundary("+y", velocity=torch.tensor([[lid, 0.0]], dtype=dt, device="cuda"))
        b.setVelocity(vel[None, ..., lo:hi, :].contiguous())
        blocks.append(b)
    if case["blocks"] > 1:
        blocks[0].ConnectBlock("+y", blocks[1], "-y", "-x")
        blocks[1].ConnectBlock("+y", blocks[0], "-y", "-x")
    dom.PrepareSolve()
    return dom


def _simulation(case, dom):
    tol = _solver_tolerance(case)
    return S.Simulation(dom, time_step=_flow_parameters(case)[3], corrector_steps=2, non_orthogonal=False,
                        advection_tol=tol[0], pressure_tol=tol[1], advect_passive_scalar=False)


def _solver_tolerance(case):
    """(advection, pressure) stopping tolerances, absolute as the criterion is.  The pressure systems of these flows
    have right-hand sides of RMS 1e-6 to 1e-4 and their adjoints of about 1: these are two to four digits below."""
    if case["dtype"] == "f64":
        return 1e-10, 1e-11
    return 1e-7, {"step": 1e-9, "batch": 1e-9, "grad": 1e-8}.get(case["kind"], 1e-7)


def _system(case, seed):
    """A pressure (cg, refine) or advection (bicg) system: ELL columns and values [n, k] in 64 bits but rounded to
    the case's precision (absent entries: the row's own column with value 0), and right-hand sides [m, n] of RMS 1."""
    g = torch.Generator().manual_seed(seed)
    dt = _DTYPE[case["dtype"]]
    verts, per = _axes(case)
    if case["ogrid"]:
        return _ogrid_system(case, g, dt)
    h = [v[1:] - v[:-1] for v in verts]
    dims = len(h)
    shape = [case["nx"], case["ny"]] + ([case["nz"]] if dims == 3 else [])
    shape = shape[::-1]
    num = torch.arange(math.prod(shape)).reshape(shape)

    def along(d, v):  # a per-axis vector as a broadcastable array
        return v.reshape([-1 if a == dims - 1 - d else 1 for a in range(dims)])

    det = torch.ones(shape, dtype=torch.float64)
    for d in range(dims):
        det = det * along(d, h[d])
    noise = torch.rand(shape, generator=g, dtype=torch.float64)
    cols, vals = [num], [torch.zeros(shape, dtype=torch.float64)]
    _, _, umax, tstep = _flow_parameters(case)
    if case["kind"] == "bicg":
        vel = _velocity(case, seed)
        visc = _flow_parameters(case)[0]
        diag = torch.ones(shape, dtype=torch.float64) / tstep
    else:
        a = tstep / (1.0 + 0.3 * noise)  # 1/A of a step: the time step damped by advection and viscosity
        diag = torch.zeros(shape, dtype=torch.float64)
    for d in range(dims):
        ax = dims - 1 - d
        alpha = det / along(d, h[d]) ** 2
        for side in (-1, 1):
            nb = torch.roll(num, -side, ax)
            inside = torch.ones(shape, dtype=torch.float64)
            if not per[d]:
                inside.select(ax, 0 if side < 0 else shape[ax] - 1).zero_()
            if case["kind"] == "bicg":
                flux = 0.25 * side * (vel[d] * det / along(d, h[d]) + torch.roll(vel[d] * det / along(d, h[d]), -side, ax))
                diff = 0.5 * visc * (alpha + torch.roll(alpha, -side, ax))
                off = (flux - diff) * inside / det
                diag = diag + ((flux + diff) * inside + 2 * visc * alpha * (1 - inside)) / det
            else:
                off = 0.5 * (alpha * a + torch.roll(alpha * a, -side, ax)) * inside
                off = off.to(dt).double()
                diag = diag - off
            cols.append(torch.where(inside > 0, nb, num))
            vals.append(off)
    vals[0] = diag
    col = torch.stack([c.reshape(-1) for c in cols], 1)
    val = torch.stack([v.reshape(-1) for v in vals], 1).to(dt).double()
    n = num.numel()
    if case["kind"] == "bicg":
        rhs = vel.reshape(dims, n) / tstep
    else:
        u = _velocity(case, seed + 1)
        rhs = torch.zeros(shape, dtype=torch.float64)
        for d in range(dims):
            ax = dims - 1 - d
            f = u[d] * det / along(d, h[d])
            up = 0.5 * (f + torch.roll(f, -1, ax))
            if not per[d]:
                up.select(ax, shape[ax] - 1).zero_()
            rhs = rhs + up - torch.roll(up, 1, ax)
        rhs = rhs.reshape(1, n)
        rhs = rhs - rhs.mean()
    rhs = rhs / rhs.pow(2).mean().sqrt()
    return col, val, rhs.to(dt).double()


def _ogrid_system(case, g, dt):
    """Pressure system of an O-grid around a cylinder: four blocks of nx cells along the angle and ny along the
    radius (clustered at the cylinder), numbered block by block, walls inside and outside."""
    nx, ny = case["nx"], case["ny"]
    r = 0.5 + 4.5 * (1.0 - torch.tanh(1.9 * (1.0 - torch.linspace(0, 1, ny + 1, dtype=torch.float64))) / math.tanh(1.9))
    dr, rc = r[1:] - r[:-1], 0.5 * (r[1:] + r[:-1])
    dth = 2 * math.pi / (4 * nx)
    num = torch.arange(4 * nx * ny).reshape(4, ny, nx).permute(1, 0, 2).reshape(ny, 4 * nx)
    a = 0.01 / (1.0 + 0.3 * torch.rand([ny, 4 * nx], generator=g, dtype=torch.float64))
    w_t = (dr / (rc * dth))[:, None] * a   # angular coefficient of a cell
    w_r = (rc * dth / dr)[:, None] * a     # radial coefficient
    cols, vals = [num], [None]
    diag = torch.zeros([ny, 4 * nx], dtype=torch.float64)
    for ax, w in ((1, w_t), (0, w_r)):
        for side in (-1, 1):
            inside = torch.ones([ny, 4 * nx], dtype=torch.float64)
            if ax == 0:
                inside[0 if side < 0 else ny - 1] = 0
            off = (0.5 * (w + torch.roll(w, -side, ax)) * inside).to(dt).double()
            diag = diag - off
            cols.append(torch.where(inside > 0, torch.roll(num, -side, ax), num))
            vals.append(off)
    vals[0] = diag
    order = torch.argsort(num.reshape(-1))
    col = torch.stack([c.reshape(-1) for c in cols], 1)[order]
    val = torch.stack([v.reshape(-1) for v in vals], 1).to(dt).double()[order]
    u = torch.randn([ny, 4 * nx], generator=g, dtype=torch.float64)
    for _ in range(6):
        u = 0.5 * u + 0.25 * (torch.roll(u, 1, 1) + torch.roll(u, -1, 1))
    rhs = (u - torch.roll(u, 1, 1)).reshape(-1)[order] + 0.05 * torch.randn(4 * nx * ny, generator=g, dtype=torch.float64)
    rhs = (rhs - rhs.mean())[None]
    rhs = rhs / rhs.pow(2).mean().sqrt()
    return col, val, rhs.to(dt).double()


def _csr(col, val, dt):
    """CSR tensors on the GPU (rows sorted by column, absent entries dropped)."""
    n = col.size(0)
    keep = torch.ones_like(col, dtype=torch.bool)
    keep[:, 1:] = col[:, 1:] != torch.arange(n)[:, None]
    big = torch.where(keep, col, torch.full_like(col, n))
    big, order = torch.sort(big, 1)
    val = torch.gather(val, 1, order)
    keep = big < n
    row = torch.zeros(n + 1, dtype=torch.int32)
    row[1:] = torch.cumsum(keep.sum(1), 0)
    return P.CSRmatrix(val[keep].to(dt).cuda(), big[keep].to(torch.int32).cuda(), row.cuda())


# --------------------------------------------------------------------------------------------------------------
# prepare, run
# --------------------------------------------------------------------------------------------------------------

def _batch_members(case):
    """Sizes and viscosities (log-uniform) of the batch's cavities."""
    g = torch.Generator().manual_seed(1000 + case["seed0"])
    lo, hi = math.log(case["lo"]), math.log(case["hi"])
    out = []
    for i in range(case["count"]):
        s, v = torch.rand(2, generator=g, dtype=torch.float64).tolist()
        n = int(round(math.exp(lo + (hi - lo) * s)))
        out.append(dict(kind="step", nx=n, ny=n, nz=0, flow="cavity", blocks=1, steps=1, dtype=case["dtype"],
                        visc=10.0 ** (-3 + 2 * v), dt=0.4 / case["hi"]))
    return out


def prepare(case, seed):
    kind = case["kind"]
    dt = _DTYPE[case["dtype"]]
    if kind == "batch":
        members = _batch_members(case)
        doms = [_domain(m, seed + i, "cavity%d" % i) for i, m in enumerate(members)]
        tol = _solver_tolerance(case)
        sims = [S.Simulation(d, time_step=m["dt"], corrector_steps=2, non_orthogonal=False, advection_tol=tol[0],
                             pressure_tol=tol[1], advect_passive_scalar=False) for d, m in zip(doms, members)]
        batch = SimulationBatch(sims)
        batch.tune()
        u0 = [d.getBlock(0).velocity.clone() for d in doms]
        return dict(case=case, batch=batch, doms=doms, u0=u0)
    if kind in ("step", "grad"):
        dom = _domain(case, seed)
        sim = _simulation(case, dom)
        u0 = [b.velocity.clone() for b in dom.getBlocks()]
        st = dict(case=case, dom=dom, sim=sim, u0=u0)
        if kind == "grad":
            sim.defer_solver_checks = True
            t = _target(case, seed).to(dtype=dt, device="cuda")
            st["target"] = [t[None, ..., lo:hi, :].contiguous() for lo, hi in _block_slices(case)]
            st["force"] = [torch.zeros_like(u) for u in u0]
        return st
    col, val, rhs = _system(case, seed)
    b = rhs.reshape(-1).to(dt).cuda()
    return dict(case=case, A=_csr(col, val, dt), b=b)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "batch":
        torch._foreach_copy_([d.getBlock(0).velocity for d in state["doms"]], state["u0"])
        state["batch"].step()
        # the samples of a data set go into one buffer per field
        return [torch.cat([d.getBlock(0).velocity.reshape(-1) for d in state["doms"]]),
                torch.cat([d.getBlock(0).pressure.reshape(-1) for d in state["doms"]])]
    if kind == "step":
        blocks = state["dom"].getBlocks()
        for b, u in zip(blocks, state["u0"]):
            b.velocity.copy_(u)
        if not state["sim"].run(case["steps"]):
            raise RuntimeError("simulation failed")
        return [b.velocity for b in blocks] + [b.pressure for b in blocks]
    if kind == "grad":
        return _run_grad(state)
    tol = _solver_tolerance(case)
    n = state["A"].getRows()
    if kind == "refine":
        x = torch.zeros(n, dtype=torch.float64, device="cuda")
        info = P.SolveLinearRefined(state["A"], state["b"], x, 5000, 1e-5, 1e-10)
        return x - x.mean()
    x = torch.zeros_like(state["b"])
    infos = P.SolveLinear(state["A"], state["b"], x, maxIterations=5000, tolerance=tol[0] if kind == "bicg" else tol[1],
                          useBiCG=kind == "bicg", BiCGwithPreconditioner=False)
    if not all(i.converged for i in infos):
        raise RuntimeError("solve did not converge")
    return x if kind == "bicg" else x - x.mean()


def _run_grad(state):
    sim, dom = state["sim"], state["dom"]
    blocks = dom.getBlocks()
    u = [t.clone().requires_grad_(True) for t in state["u0"]]
    f = [t.clone().requires_grad_(True) for t in state["force"]]
    for b, ub, fb in zip(blocks, u, f):
        b.setVelocity(ub)
        b.setVelocitySource(fb)
    dom.UpdateDomainData()
    out = CK.rollout(sim, state["case"]["steps"], params=f, checkpoint=True)
    loss = sum(((o - t) ** 2).sum() for o, t in zip(out, state["target"]))
    loss.backward()
    sim.flush_solver_checks()
    return [o.detach() for o in out] + [t.grad for t in u] + [t.grad for t in f]


# --------------------------------------------------------------------------------------------------------------
# work, tolerance
# --------------------------------------------------------------------------------------------------------------

def work(case):
    """The least a pass can move and compute.  An iterative solve has to read its matrix and right-hand side and
    write its solution at least once; a step reads the metrics, velocity and boundary data and writes velocity and
    pressure; a gradient pass adds its mirrored traffic.  Iterations kept on chip need no memory traffic, so no
    iteration count enters the bytes; the flops count the products of about one iteration per grid line across the
    longest axis, as an unpreconditioned Krylov solve needs."""
    s = 4 if case["dtype"] == "f32" else 8
    if case["kind"] == "batch":
        ws = [work(m) for m in _batch_members(case)]
        return {"bytes": sum(w["bytes"] for w in ws), "flops": sum(w["flops"] for w in ws)}
    n = _cells(case)
    dims = 3 if case["nz"] else 2
    nz = 2 * dims + 1
    iters = max(case["nx"], case["ny"], case["nz"]) * (2 if case.get("ogrid") else 1)
    spmv = 2 * nz * n
    if case["kind"] == "cg":
        return {"bytes": n * (nz * (s + 4) + 4 + 2 * s), "flops": iters * (spmv + 12 * n)}
    if case["kind"] == "refine":
        return {"bytes": n * (nz * (s + 4) + 4 + s + 8), "flops": 2 * iters * (spmv + 12 * n)}
    if case["kind"] == "bicg":
        return {"bytes": n * (nz * (s + 4) + 4 + 2 * dims * s), "flops": 10 * dims * (2 * spmv + 20 * n)}
    # a step: metrics (2 D^2 + 1), velocity in, velocity and pressure out
    step = {"bytes": n * s * (2 * dims * dims + 1 + 2 * dims + 1),
            "flops": 2 * iters * (spmv + 12 * n) + 10 * dims * (2 * spmv + 20 * n)}
    k = case["steps"] * (1 if case["kind"] == "step" else 3)
    extra = 0 if case["kind"] == "step" else n * s * 4 * dims
    return {"bytes": k * step["bytes"] + extra, "flops": k * step["flops"]}


def tolerance(case):
    """Measured with the solvers' sums in another order and on other kernels, times about four.  The largest part is
    a solve that stops one iteration earlier or later: its last iteration moves the solution by about a tenth of the
    distance from the converged one (pressure of a box or batch step: 5e-4, a gradient: 3e-5, FP64: 8e-7)."""
    if case["dtype"] == "f64":
        return {"rel": {"step": 4e-7, "grad": 4e-9, "cg": 4e-10, "bicg": 4e-9}[case["kind"]]}
    return {"step": {"rel": 2e-4, "max": 1e-3}, "batch": {"rel": 2e-4, "max": 1e-3}, "grad": {"rel": 2e-5, "max": 3e-4},
            "cg": {"rel": 1e-5, "max": 2e-4}, "bicg": {"rel": 1e-6, "max": 2e-5}, "refine": {"rel": 1e-9}}[case["kind"]]


# --------------------------------------------------------------------------------------------------------------
# the same in 64 bits on whole arrays
# --------------------------------------------------------------------------------------------------------------

def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _cg64(mv, b, project):
    """Converged CG in 64 bits on the array b (project: the constant is in the null space)."""
    x = torch.zeros_like(b)
    r = b - b.mean() if project else b.clone()
    p = r.clone()
    rho = (r * r).sum()
    stop = 1e-13 * float(rho.sqrt())
    if stop == 0.0:
        return x
    for it in range(20000):
        q = mv(p)
        alpha = rho / (p * q).sum()
        x = x + alpha * p
        r = r - alpha * q
        if project:
            r = r - r.mean()
        new = (r * r).sum()
        p = r + (new / rho) * p
        rho = new
        if it % 20 == 19 and float(rho.sqrt()) < stop:
            break
    return x - x.mean() if project else x


def _bicg64(mv, b):
    """Converged BiCGStab in 64 bits."""
    x = torch.zeros_like(b)
    r = b.clone()
    h = r.clone()
    rho = (h * r).sum()
    stop = 1e-13 * float(r.norm())
    if stop == 0.0:
        return x
    p = r.clone()
    for it in range(2000):
        v = mv(p)
        alpha = rho / (h * v).sum()
        s = r - alpha * v
        if float(s.norm()) < stop:
            return x + alpha * p
        t = mv(s)
        omega = (t * s).sum() / (t * t).sum()
        x = x + alpha * p + omega * s
        r = s - omega * t
        if float(r.norm()) < stop:
            return x
        new = (h * r).sum()
        p = r + (new / rho) * (alpha / omega) * (p - omega * v)
        rho = new
    return x


class _Implicit(torch.autograd.Function):
    """Zero with the derivative of a linear solve: the residual's gradient is the transposed solve of the output's."""

    @staticmethod
    def forward(ctx, residual, transposed):
        ctx.transposed = transposed
        return torch.zeros_like(residual)

    @staticmethod
    def backward(ctx, g):
        return ctx.transposed(g), None


class _Step64:
    """The PISO step of one tensor-product grid on arrays [(nz,) ny, nx] (blocks joined along y are one array)."""

    def __init__(self, case):
        verts, self.per = _rounded_axes(case)
        dev = _device()
        verts = [v.double().to(dev) for v in verts]
        self.D = len(verts)
        visc, self.lid, _, dt = _flow_parameters(case)
        dtype = _DTYPE[case["dtype"]]
        # scalars as the framework holds them
        self.nu = float(torch.tensor(case.get("visc", visc), dtype=dtype))
        self.dt = float(torch.tensor(case.get("dt", dt), dtype=dtype))
        self.shape = [v.numel() - 1 for v in verts][::-1]
        h = [v[1:] - v[:-1] for v in verts]
        h = [w.reshape([-1 if a == self.D - 1 - d else 1 for a in range(self.D)]).expand(self.shape)
             for d, w in enumerate(h)]
        self.h = h
        self.det = math.prod(h[1:], start=h[0]) if self.D > 1 else h[0]
        self.alpha = [self.det / w ** 2 for w in h]
        self.mask = {}
        for d in range(self.D):
            for side in (-1, 1):
                m = torch.ones(self.shape, dtype=torch.float64, device=dev)
                if not self.per[d]:
                    m.select(self.D - 1 - d, 0 if side < 0 else -1).zero_()
                self.mask[d, side] = m
        # wall source of a moving +y wall
        self.wall = [torch.zeros(self.shape, dtype=torch.float64, device=dev) for _ in range(self.D)]
        if self.lid:
            self.wall[0] = (1 - self.mask[1, 1]) * self.lid * self.nu * 2 * self.alpha[1] / self.det

    def nb(self, q, d, side):
        return torch.roll(q, -side, self.D - 1 - d)

    def apply(self, diag, off, v):
        y = diag * v
        for (d, s), c in off.items():
            y = y + c * self.nb(v, d, s)
        return y

    def apply_t(self, diag, off, v):
        y = diag * v
        for (d, s), c in off.items():
            y = y + self.nb(c * v, d, -s)
        return y

    def solve(self, diag, off, b, singular=False):
        """x with diag/off x = b, differentiable in all three."""
        with torch.no_grad():
            dd, oo = diag.detach(), {k: c.detach() for k, c in off.items()}
            sign = -1.0 if singular else 1.0
            if singular:
                x = -_cg64(lambda v: sign * self.apply(dd, oo, v), b.detach(), True)
            else:
                x = _bicg64(lambda v: self.apply(dd, oo, v), b.detach())

        def transposed(g):
            if singular:
                return -_cg64(lambda v: sign * self.apply(dd, oo, v), g, True)
            return _bicg64(lambda v: self.apply_t(dd, oo, v), g)
        if not (torch.is_grad_enabled() and (b.requires_grad or diag.requires_grad)):
            return x
        return x + _Implicit.apply(b - self.apply(diag, off, x), transposed)

    def step(self, u, src):
        D, det, dt = self.D, self.det, self.dt
        U = [u[d] * det / self.h[d] for d in range(D)]
        diag = det / dt
        off = {}
        for d in range(D):
            for s in (-1, 1):
                m = self.mask[d, s]
                flux = 0.25 * s * (U[d] + self.nb(U[d], d, s)) * m
                diff = 0.5 * self.nu * (self.alpha[d] + self.nb(self.alpha[d], d, s)) * m
                diag = diag + flux + diff + 2 * self.nu * self.alpha[d] * (1 - m)
                off[d, s] = (flux - diff) / det
        A = diag / det
        const = [u[d] / dt + self.wall[d] + src[d] for d in range(D)]
        v = [self.solve(A, off, const[d]) for d in range(D)]
        pdiag, poff = 0, {}
        for d in range(D):
            for s in (-1, 1):
                w = self.alpha[d] / A
                c = 0.5 * (w + self.nb(w, d, s)) * self.mask[d, s]
                poff[d, s] = c
                pdiag = pdiag - c
        zero = torch.zeros_like(A)
        p = None
        for _ in range(2):
            hbya = [(const[d] - self.apply(zero, off, v[d])) / A for d in range(D)]
            div = 0
            for d in range(D):
                W = hbya[d] * det / self.h[d]
                for s in (-1, 1):
                    div = div + 0.5 * s * (W + self.nb(W, d, s)) * self.mask[d, s]
            p = self.solve(pdiag, poff, div, singular=True)
            p = p - p.mean()
            v = []
            for d in range(D):
                hi = self.mask[d, 1] * self.nb(p, d, 1) + (1 - self.mask[d, 1]) * p
                lo = self.mask[d, -1] * self.nb(p, d, -1) + (1 - self.mask[d, -1]) * p
                fac = 0.5 + 0.5 * ((1 - self.mask[d, 1]) + (1 - self.mask[d, -1]))
                v.append(hbya[d] - (hi - lo) * fac / self.h[d] / A)
        return v, p


def _split(case, arrays):
    """[D, ...] components as the blocks' tensors [1, D, ...]."""
    t = torch.stack(list(arrays))[None]
    return [t[..., lo:hi, :] for lo, hi in _block_slices(case)]


def _exact_step(case, seed):
    m = _Step64(case)
    u = _velocity(case, seed).to(_DTYPE[case["dtype"]]).double().to(_device())
    u = [u[d] for d in range(m.D)]
    zero = [torch.zeros_like(u[0])] * m.D
    with torch.no_grad():
        for _ in range(case["steps"]):
            u, p = m.step(u, zero)
    return _split(case, u) + _split(case, [p])


def _exact_grad(case, seed):
    m = _Step64(case)
    dtype = _DTYPE[case["dtype"]]
    u0 = _velocity(case, seed).to(dtype).double().to(_device()).requires_grad_(True)
    f = torch.zeros_like(u0).requires_grad_(True)
    t = _target(case, seed).to(dtype).double().to(_device())
    u = [u0[d] for d in range(m.D)]
    for _ in range(case["steps"]):
        u, _ = m.step(u, [f[d] for d in range(m.D)])
    loss = sum(((o - w) ** 2).sum() for o, w in zip(_split(case, u), _split(case, list(t))))
    loss.backward()
    det = lambda x: [x[d].detach() for d in range(m.D)]  # noqa: E731
    return _split(case, det(u)) + _split(case, det(u0.grad)) + _split(case, det(f.grad))


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        each = [_exact_step(m, seed + i) for i, m in enumerate(_batch_members(case))]
        return [torch.cat([e[k].reshape(-1) for e in each]) for k in (0, 1)]
    if kind == "step":
        return _exact_step(case, seed)
    if kind == "grad":
        return _exact_grad(case, seed)
    col, val, rhs = (t.to(_device()) for t in _system(case, seed))
    mv = lambda v: (val * v[col]).sum(1)  # noqa: E731
    if kind == "bicg":
        return torch.cat([_bicg64(mv, b) for b in rhs])
    return -_cg64(lambda v: -mv(v), rhs[0], True)
