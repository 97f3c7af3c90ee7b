"""Performance cases of the solver kernels: what a user's program has the
framework do, through its public entry points, over the range in use.

A case is one complete piece of a user's run: take initial conditions (or a
saved state), find the stable time step, advance a number of steps on the
device and read the solution back -- the loop of a simulation between two
plots.  The kinds:

  cell      one cell through the per-cell plugin surface (host arrays in and
            out, one call per kernel): the drop-in use from a host engine
  dg        a regular mesh of ADER-DG cells resident on the device
  ensemble  independent small grids of several orders in shared launches
  limiter   limiting ADER-DG on an adaptive mesh (refined shell around a
            Sod sphere, MUSCL-Hancock subcells on the finest level)
  fv        a mesh of finite-volume patches (2D Godunov, 3D MUSCL-Hancock)
  transfer  batched prolongation and restriction between mesh levels

`exact` recomputes the results with plain torch in 64 bits from the
definition of the schemes.
"""
import math

import numpy as np
import torch

import exahype_amd as E

V = 5
GAMMA = 1.4
CFL = 0.9
PRECISIONS = {"fp64": E.PREC_FP64, "fp32": E.PREC_FP32}
VELOCITY = (0.3, -0.7, 0.5)  # of the linear-advection PDE


# ---------------------------------------------------------------------------
# cases

def listed():
    return [
        # one cell, every kernel a separate call on host arrays: what a host
        # engine pays per cell when it calls the virtuals directly
        dict(name="cell_n3", kind="cell", order=3),
        # a small mesh: launches and gaps between them count
        dict(name="dg_n3_9_fp64", kind="dg", order=3, nx=9, ny=9, nz=9, precision="fp64", steps=60, pde="euler",
             restart=False),
        # the ordinary production order and mesh, mixed-precision predictor
        dict(name="dg_n5_27_mixed", kind="dg", order=5, nx=27, ny=27, nz=27, precision="fp32", steps=60, pde="euler",
             restart=False),
        # the same order, a large mesh with odd sides, plain double precision
        dict(name="dg_n5_45x44x43_fp64", kind="dg", order=5, nx=45, ny=44, nz=43, precision="fp64", steps=60,
             pde="euler", restart=False),
        # a high order from a saved state (restart): upload, steps, download
        dict(name="dg_n7_18x19x20_fp64", kind="dg", order=7, nx=18, ny=19, nz=20, precision="fp64", steps=40,
             pde="euler", restart=True),
        # the highest order, mixed precision
        dict(name="dg_n9_15x16x17_mixed", kind="dg", order=9, nx=15, ny=16, nz=17, precision="fp32", steps=20,
             pde="euler", restart=False),
        # a PDE with a non-conservative product: the kernels that a project's
        # own PDE runs on
        dict(name="dg_n4_ncp_25x26x27", kind="dg", order=4, nx=25, ny=26, nz=27, precision="fp64", steps=40,
             pde="advection_ncp", restart=False),
        # parameter study: independent grids of orders 3..7
        dict(name="ensemble_20", kind="ensemble", members=20, side=18, precision="fp32", steps=20),
        # adaptive mesh with shocks: predictor, hanging faces, limiter
        dict(name="limiter_n5_9_3lev", kind="limiter", order=5, base=9, levels=3, precision="fp64", steps=15),
        # the EulerFV demonstrator: 81 x 81 patches of 10 x 10 volumes
        dict(name="fv2d_godunov_81x81", kind="fv", dim=2, patch=10, nx=81, ny=81, nz=1, steps=200),
        # second-order finite volumes on the limiter's subcell patches
        dict(name="fv3d_muscl_12x13x14", kind="fv", dim=3, patch=11, nx=12, ny=13, nz=14, steps=60),
        # level transfers of a mesh change
        dict(name="transfer_n5_12", kind="transfer", order=5, n=12),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["cell", "dg", "dg", "dg", "dg", "ensemble", "limiter", "fv", "fv", "transfer"])
    if kind == "cell":
        return dict(kind="cell", order=rng.randint(1, 9))
    if kind == "dg":
        order = rng.randint(1, 9)
        # up to as many nodes as the large listed mesh has
        most = (45 * 44 * 43 * 6 ** 3 / (order + 1) ** 3 * (1.0 if order < 7 else 0.4)) ** (1 / 3)
        nx, ny, nz = (_log(rng, 4, max(5, min(60, most))) for _ in range(3))
        pde = "advection_ncp" if order <= 7 and rng.random() < 0.2 else "euler"
        precision = "fp64" if pde != "euler" else rng.choice(["fp64", "fp32"])
        return dict(kind="dg", order=order, nx=nx, ny=ny, nz=nz, precision=precision, steps=rng.randint(10, 40),
                    pde=pde, restart=rng.random() < 0.3)
    if kind == "ensemble":
        return dict(kind="ensemble", members=rng.randint(2, 20), side=rng.randint(6, 18),
                    precision=rng.choice(["fp64", "fp32"]), steps=rng.randint(5, 20))
    if kind == "limiter":
        return dict(kind="limiter", order=rng.randint(3, 5), base=rng.randint(5, 9), levels=rng.randint(1, 3),
                    precision=rng.choice(["fp64", "fp32"]), steps=rng.randint(3, 15))
    if kind == "fv":
        if rng.random() < 0.5:
            return dict(kind="fv", dim=2, patch=rng.randint(4, 20), nx=_log(rng, 3, 60), ny=_log(rng, 3, 60), nz=1,
                        steps=rng.randint(20, 200))
        return dict(kind="fv", dim=3, patch=2 * rng.randint(1, 6) + 1, nx=_log(rng, 3, 12), ny=_log(rng, 3, 12),
                    nz=_log(rng, 3, 12), steps=rng.randint(10, 60))
    order = rng.randint(2, 7)
    return dict(kind="transfer", order=order, n=_log(rng, 3, int(12 * 6 / (order + 1))))


# ---------------------------------------------------------------------------
# inputs

def _modes(rng, **kw):
    return dict(rho_inf=1.0, p_inf=1.0, amp=1e-2, nmodes=8, k=rng.integers(1, 4, size=(8, 3)).astype(float),
                a=rng.uniform(-1, 1, 8), phi=rng.uniform(0, 2 * np.pi, 8), **kw)


def _vortex(rng):
    """An isentropic vortex on a drifting background plus eight density modes."""
    return _modes(rng, xc=tuple(rng.uniform(0.3, 0.7, 3)), L=0.1, eps=float(rng.uniform(2, 5)),
                  uinf=tuple(rng.uniform(-1, 1, 3)))


def _inputs(case, seed):
    """The numbers of a case's initial state, shared by the run and `exact`."""
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "dg" and case["pde"] != "euler":
        return dict(nmodes=2, k=rng.integers(0, 2, size=(2, 3)) + [[1, 0, 0], [0, 1, 0]], a=rng.uniform(0.05, 0.2, 2),
                    phi=rng.uniform(0, 2 * np.pi, 2), uinf=VELOCITY)
    if kind in ("cell", "dg"):
        return _vortex(rng)
    if kind == "ensemble":
        out = []
        for i in range(case["members"]):
            # every order occurs with every size
            side = max(4, int(round(case["side"] * (0.5, 0.75, 1.0)[i % 3])))
            out.append(dict(order=3 + i % 5, cells=(side, side, side), gamma=float(rng.uniform(1.3, 1.67)),
                            ic=_vortex(rng)))
        return out
    if kind == "limiter":
        # a Sod sphere whose surface lies inside the refined shell
        return dict(xc=tuple(0.5 + rng.uniform(-0.005, 0.005, 3)), r0=0.25, rho_in=1.0,
                    p_in=float(rng.uniform(0.9, 1.1)), rho_out=0.125, p_out=0.1)
    if kind == "fv":
        xc = tuple(rng.uniform(0.3, 0.7, 3)[:case["dim"]]) + (0.0,) * (3 - case["dim"])  # a 2D domain lies at z = 0
        return dict(xc=xc, L=0.01 if case["dim"] == 2 else 0.03, amp=0.5, rho_inf=1.0, p_inf=1.0,
                    uinf=tuple(rng.uniform(0.05, 0.3, 3)))
    raise ValueError(kind)


def _ic(case, seed):
    kind = case["kind"]
    k = {"limiter": 1, "fv": 5}.get(kind, 3 if case.get("pde") == "advection_ncp" else 0)
    return E.make_ic(k, **_inputs(case, seed))


def _solver(case):
    if case.get("pde", "euler") == "euler":
        return E.ADERDGSolver(case["order"], precision=PRECISIONS[case["precision"]], cfl=CFL, gamma=GAMMA)
    return E.ADERDGSolver(case["order"], pde=E.PDE_ADVECTION_NCP, velocity=VELOCITY, cfl=CFL)


class _View:
    """A DeviceArray for torch.as_tensor, without a copy."""

    def __init__(self, a):
        self.array = a
        self.__cuda_array_interface__ = dict(shape=(a.n,), typestr="<f8", data=(a.ptr.value, False), version=3)


def _tensor(a):
    t = torch.as_tensor(_View(a), device="cuda")
    t.array = a  # the memory lives as long as the tensor
    return t


def _transfer_lists(case):
    """Children of every coarse cell one level down: offsets and sub-cell index."""
    blk = (case["order"] + 1) ** 3 * V
    child = np.arange(27 * case["n"] ** 3)
    sub = child % 27
    return E.amr_transfer_array(child * blk, child // 27 * blk, 1, np.stack([sub % 3, sub // 3 % 3, sub // 9], axis=1))


def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=case)
    if kind == "cell":
        s = st["solver"] = E.ADERDGSolver(case["order"], cfl=CFL, gamma=GAMMA)
        st["dx"] = np.array([0.125, 0.1, 0.1])
        st["luh"] = s.adjustSolution((0.5, 0.55, 0.45), st["dx"], 0.0, _ic(case, seed))
        st["dt"] = s.stableTimeStepSize(st["luh"], st["dx"])
    elif kind == "dg":
        st["solver"] = _solver(case)
        g = st["grid"] = E.Grid(st["solver"], case["nx"], case["ny"], case["nz"])
        g.use_graph(True)
        st["ic"] = _ic(case, seed)
        if case["restart"]:
            g.set_initial_conditions(st["ic"])
            st["saved"] = g.download()
    elif kind == "ensemble":
        ms = _inputs(case, seed)
        st["grid"] = E.Ensemble(ms, precision=PRECISIONS[case["precision"]], cfl=CFL)
        st["ics"] = [E.make_ic(0, **m["ic"]) for m in ms]
    elif kind == "limiter":
        st["solver"] = _solver(case)
        st["ic"] = _ic(case, seed)
        g = st["grid"] = E.AMRGrid(st["solver"], E.amr_config(case["base"], case["levels"], (0.5, 0.5, 0.5), 0.25,
                                                              (0.06, 0.031)))
        g.use_graph(True)
    elif kind == "fv":
        scheme = E.FV_GODUNOV if case["dim"] == 2 else E.FV_MUSCLHANCOCK
        st["solver"] = E.FiniteVolumesSolver(case["dim"], case["patch"], scheme=scheme, cfl=CFL, gamma=GAMMA)
        st["grid"] = E.FVGrid(st["solver"], case["nx"], case["ny"], case["nz"])
        st["ic"] = _ic(case, seed)
    else:
        nc, blk = case["n"] ** 3, (case["order"] + 1) ** 3 * V
        rng = np.random.default_rng(seed)
        st["coarse"] = E.DeviceArray(1.0 + rng.random(nc * blk))
        st["fine"], st["back"] = E.DeviceArray(27 * nc * blk), E.DeviceArray(nc * blk)
        st["fine_t"] = _tensor(st["fine"])
        st["back_t"] = _tensor(st["back"])
        st["list"] = _transfer_lists(case)
    return st


# ---------------------------------------------------------------------------
# one pass

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "cell":
        s, dx, dt = state["solver"], state["dx"], state["dt"]
        pred = s.spaceTimePredictor(state["luh"], dx, dt)
        lduh = s.volumeIntegral(pred["lFhi"], dx)
        # the cell is its own neighbour across every face
        q, f = pred["lQhbnd"].reshape(6, -1), pred["lFhbnd"].reshape(6, -1)
        flux = np.empty_like(f)
        for d in range(3):
            flux[2 * d + 1], flux[2 * d] = s.riemannSolver(f[2 * d + 1], f[2 * d], q[2 * d + 1], q[2 * d], dt, d)
        lduh = s.surfaceIntegral(lduh, flux, dx)
        luh = s.solutionUpdate(state["luh"], lduh, dt)
        return dict(lQi=pred["lQi"], lQhi=pred["lQhi"], lFhi=pred["lFhi"], lQhbnd=pred["lQhbnd"],
                    lFhbnd=pred["lFhbnd"], flux=flux, lduh=lduh, luh=luh, dt=s.stableTimeStepSize(luh, dx))
    if kind == "transfer":
        fine, back = state["fine"], state["back"]
        state["back_t"].zero_()  # restrictions add
        torch.cuda.current_stream().synchronize()  # the library works on streams of its own
        E.amrProlongationBatched(3, case["order"], V, fine, state["coarse"], state["list"])
        E.amrRestrictionBatched(3, case["order"], V, back, fine, state["list"])
        return dict(fine=state["fine_t"], back=state["back_t"])
    g = state["grid"]
    if kind == "ensemble":
        g.set_initial_conditions(state["ics"])
        g.compute_dt()
        g.step(case["steps"])
        t, dt = g.sync()
        return dict(t=t, dt=dt, u=[g.download(i) for i in range(g.n)])
    if case.get("restart"):
        g.upload(state["saved"])
    else:
        g.set_initial_conditions(state["ic"])
    t0 = 0.0 if kind == "limiter" else g.sync()[0]  # a grid's time runs on
    g.compute_dt()
    g.step(case["steps"])
    t, dt = g.sync()[:2]
    if kind == "fv":
        u = g.download().reshape((-1,) + (g.solver.side,) * case["dim"] + (V,))
        inner = slice(g.solver.ghost, g.solver.ghost + case["patch"])
        u = u[:, inner, inner] if case["dim"] == 2 else u[:, inner, inner, inner]
        return dict(t=t - t0, dt=dt, u=u)
    if kind == "limiter":
        return dict(dt=dt, u=g.download(), status=g.limiter_status())
    return dict(t=t - t0, dt=dt, u=g.download())


# ---------------------------------------------------------------------------
# what a pass cannot do without

def _dg_work(order, cells, steps, sweeps=3.0):
    """Bytes: the state read and written once per step and read back once.
    Flops: Picard sweeps (three are what these time steps take; the first
    starts from data constant in time, so one time level suffices), time
    averages, volume and surface integral, face extrapolation."""
    B = order + 1
    level = 6 * V * B ** 4 + B ** 3 * 65  # contractions, flux and sums at one time level
    sweep = (sweeps - 1) * (B * level + 2 * V * B ** 5) + level
    flops = sweep + 14 * V * B ** 4 + 36 * V * B ** 3
    return cells * (16.0 * steps + 8) * V * B ** 3, cells * steps * flops


def work(case):
    kind = case["kind"]
    if kind == "cell":
        B = case["order"] + 1
        b = 8.0 * V * (B ** 4 + 3 * B ** 3 + 4 * B ** 3 + 18 * B ** 2)
        f = _dg_work(case["order"], 1, 1)[1]
    elif kind == "dg":
        b, f = _dg_work(case["order"], case["nx"] * case["ny"] * case["nz"], case["steps"])
    elif kind == "ensemble":
        b = f = 0.0
        for i in range(case["members"]):
            x = _dg_work(3 + i % 5, round(case["side"] * (0.5, 0.75, 1.0)[i % 3]) ** 3, case["steps"])
            b, f = b + x[0], f + x[1]
    elif kind == "limiter":
        # leaves of the unrefined mesh times the growth by the shell
        cells = case["base"] ** 3 * (1, 5, 40)[case["levels"] - 1]
        b, f = _dg_work(case["order"], cells, case["steps"], sweeps=2.0)
    elif kind == "fv":
        n = case["nx"] * case["ny"] * case["nz"] * case["patch"] ** case["dim"]
        b = n * V * (16.0 * case["steps"] + 8)
        f = n * case["steps"] * (2 * 110.0 if case["dim"] == 2 else 6 * 40 + 3 * 150.0)
    else:
        n, B = case["n"] ** 3, case["order"] + 1
        b = 8.0 * n * V * B ** 3 * (27 + 1) * 2
        f = 27.0 * n * 2 * 6 * V * B ** 4
    return dict(bytes=b, flops=f)


def tolerance(case):
    kind = case["kind"]
    if kind == "transfer":
        return dict(rel=1e-13, max=1e-12)
    if kind == "fv":
        return dict(rel=1e-13, max=1e-11)
    if kind == "cell":
        return dict(rel=4e-11, max=1e-9)
    if case["precision"] == "fp32":
        # FP32 sweeps before the FP64 correction sweep: 1.3e-7 from 64 bits
        return dict(rel=1e-6, max=1e-4, differ=1e-3)
    if kind == "limiter":
        # shocks, and decisions on thresholds
        return dict(rel=1e-9, max=1e-6, differ=1e-3)
    # 64-bit sums: another implementation is 1e-13 (order 3) to 2e-11 (order
    # 9) off; the Picard loop stops at a residual of 1e-7, so a cell on the
    # edge of that may take one sweep more or fewer
    return dict(rel=1e-10 if case.get("order", 9) > 7 else 4e-11, max=1e-8)


# ---------------------------------------------------------------------------
# the same results in 64 bits from plain torch

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


class _Ops:
    """Operators of the Lagrange basis through the Gauss-Legendre nodes of [0, 1]."""

    def __init__(self, order):
        x, w = np.polynomial.legendre.leggauss(order + 1)
        self.x, w = 0.5 * (x + 1.0), 0.5 * w
        c = [np.poly(np.delete(self.x, k)) for k in range(order + 1)]
        c = [p / np.polyval(p, self.x[k]) for k, p in enumerate(c)]
        left = np.array([np.polyval(p, 0.0) for p in c])
        right = np.array([np.polyval(p, 1.0) for p in c])
        # D[k][m] = phi_k'(x_m) by barycentric weights
        b = np.array([1.0 / np.prod(self.x[k] - np.delete(self.x, k)) for k in range(order + 1)])
        D = np.zeros((order + 1, order + 1))
        for k in range(order + 1):
            for m in range(order + 1):
                if k != m:
                    D[k, m] = b[k] / b[m] / (self.x[m] - self.x[k])
        D[np.arange(order + 1), np.arange(order + 1)] = -(D.sum(axis=0))
        K = D * w[None, :]
        t = lambda a: torch.tensor(np.ascontiguousarray(a), dtype=torch.float64, device=_device())  # noqa: E731
        self.B, self.w, self.left, self.right, self.K, self.D = order + 1, t(w), t(left), t(right), t(K), t(D)
        self.iK1 = t(np.linalg.inv(np.outer(right, right) - K))


def _contract(a, M, axis):
    """sum_n a[.., n at axis, ..] M[n][l]"""
    return torch.movedim(torch.movedim(a, axis, -1).contiguous() @ M, -1, axis)


def _along(v, axis, ndim):
    return v.reshape([-1 if i == axis % ndim else 1 for i in range(ndim)])


def _euler_flux(q, d, gamma):
    """Flux in direction d (0 x, 1 y, 2 z); variables along dimension 1."""
    r, m, e = q[:, 0], [q[:, 1], q[:, 2], q[:, 3]], q[:, 4]
    p = (gamma - 1) * (e - 0.5 * (m[0] ** 2 + m[1] ** 2 + m[2] ** 2) / r)
    u = m[d] / r
    f = [m[d]] + [m[i] * u for i in range(3)] + [(e + p) * u]
    f[1 + d] = f[1 + d] + p
    return torch.stack(f, 1)


def _speed(q, d, gamma):
    r, m, e = q[:, 0], [q[:, 1], q[:, 2], q[:, 3]], q[:, 4]
    p = (gamma - 1) * (e - 0.5 * (m[0] ** 2 + m[1] ** 2 + m[2] ** 2) / r)
    return (m[d] / r).abs() + torch.sqrt(gamma * p / r)


def _predict(u, dt, dx, ops, gamma, ncp):
    """(time-averaged state, time-averaged fluxes [3] or source [1], iterate):
    u [cell][V][z][y][x]; Picard sweeps until a cell's update is below 1e-7."""
    B, w = ops.B, ops.w
    q = u.unsqueeze(2).expand(-1, -1, B, -1, -1, -1).contiguous()
    base = u.unsqueeze(2) * _along(ops.left, 2, 6)
    avg = lambda a: torch.tensordot(a, w, dims=([2], [0]))  # noqa: E731
    todo = torch.arange(u.shape[0], device=u.device)
    avgs = [torch.empty_like(u) for _ in range(1 if ncp else 3)]
    for it in range(2 * B):
        old = q[todo]
        rhs = base[todo]
        fs = []
        if ncp:
            s = sum(-VELOCITY[d] / dx[d] * _contract(old, ops.D, 5 - d) for d in range(3))
            rhs = rhs + s * dt * _along(w, 2, 6)
            fs = [s]
        else:
            for d in range(3):
                f = _euler_flux(old, d, gamma)
                rhs = rhs - _contract(f, ops.K, 5 - d) / _along(w, 5 - d, 6) * _along(w, 2, 6) * (dt / dx[d])
                fs.append(f)
        new = _contract(rhs, ops.iK1.T.contiguous(), 2)
        q[todo] = new
        for a, f in zip(avgs, fs):
            a[todo] = avg(f)
        del rhs, fs
        left = ((new - old) ** 2).flatten(1).sum(1) >= 1e-14
        del new, old
        todo = todo[left]
        if not todo.numel():
            break
    return avg(q), avgs, q


def _faces(a, d, ops):
    """The traces of a [cell][V][z][y][x] on the lower and the upper face of direction d."""
    return (torch.tensordot(a, ops.left, dims=([4 - d], [0])), torch.tensordot(a, ops.right, dims=([4 - d], [0])))


def _dg_dt(u, dx, gamma, cfl, ncp):
    pnpm = (1.0, 0.33, 0.17, 0.1, 0.069, 0.045, 0.038, 0.03, 0.02, 0.015)[u.shape[-1] - 1]
    if ncp:
        return cfl * pnpm / sum(abs(VELOCITY[d]) / dx[d] for d in range(3))
    den = sum(_speed(u, d, gamma) / dx[d] for d in range(3))
    return float((cfl * pnpm / den).min())


def _dg_step(u, shape, dt, dx, ops, gamma, ncp, chunk):
    """One step of the periodic grid u [cell][V][z][y][x], cells z, y, x slowest first."""
    nz, ny, nx = shape
    w = ops.w
    new = u.clone()
    fl = [[torch.zeros((u.shape[0], V, ops.B, ops.B), dtype=u.dtype, device=u.device) for _ in range(6)]
          for _ in range(2)]
    for c in range(0, u.shape[0], chunk):
        part = slice(c, c + chunk)
        qh, fh, _ = _predict(u[part], dt, dx, ops, gamma, ncp)
        if ncp:
            new[part] += dt * fh[0]
        for d in range(3):
            fl[0][2 * d][part], fl[0][2 * d + 1][part] = _faces(qh, d, ops)
            if not ncp:
                fl[1][2 * d][part], fl[1][2 * d + 1][part] = _faces(fh[d], d, ops)
                new[part] += dt / dx[d] * _contract(fh[d], ops.K.T.contiguous(), 4 - d) / _along(w, 4 - d, 5)
    for d in range(3):
        roll = lambda a, n: torch.roll(a.reshape((nz, ny, nx) + a.shape[1:]), n, 2 - d).reshape(a.shape)  # noqa: E731
        ql, qr = fl[0][2 * d + 1], roll(fl[0][2 * d], -1)
        lo, hi = _riemann(ql, qr, fl[1][2 * d + 1], roll(fl[1][2 * d], -1), d, w, gamma, ncp)
        below = roll(hi, 1)  # flux of the lower face, from the neighbour's problem
        r, l = _along(ops.right / w, 4 - d, 5), _along(ops.left / w, 4 - d, 5)
        new -= dt / dx[d] * (lo.unsqueeze(4 - d) * r - below.unsqueeze(4 - d) * l)
    return new


def _riemann(ql, qr, fl, fr, d, w, gamma, ncp):
    """Rusanov fluxes as seen by the lower and the upper cell of a face."""
    if ncp:
        s = abs(VELOCITY[d])
        f = -0.5 * s * (qr - ql)
        p = 0.5 * VELOCITY[d] * (qr - ql)
        return f + p, f - p
    ww = w[:, None] * w[None, :]
    al, ar = (ql * ww).sum((2, 3)), (qr * ww).sum((2, 3))
    s = torch.maximum(_speed(al, d, gamma), _speed(ar, d, gamma)).reshape(-1, 1, 1, 1)
    f = 0.5 * (fl + fr) - 0.5 * s * (qr - ql)
    return f, f


def _start(ins, x, y, z, gamma):
    """The initial state at points: [V][...]"""
    if "L" not in ins:  # sine modes of the advection equation
        s = sum(float(a) * torch.sin(2 * math.pi * (float(k[0]) * x + float(k[1]) * y + float(k[2]) * z) + float(p))
                for a, k, p in zip(ins["a"], ins["k"], ins["phi"]))
        return torch.stack([1.0 + (v + 1) * s for v in range(V)])
    one = torch.ones_like(x)
    if "eps" in ins:
        rx, ry = ((x - torch.floor(x)) - ins["xc"][0]) / ins["L"], ((y - torch.floor(y)) - ins["xc"][1]) / ins["L"]
        r2 = rx * rx + ry * ry
        du = ins["eps"] / (2 * math.pi) * torch.exp(0.5 * (1 - r2))
        T = 1 - (gamma - 1) * ins["eps"] ** 2 / (8 * gamma * math.pi ** 2) * torch.exp(1 - r2)
        rho, p = T ** (1 / (gamma - 1)), T ** (gamma / (gamma - 1))
        vel = [ins["uinf"][0] - du * ry, ins["uinf"][1] + du * rx, ins["uinf"][2] * one]
        rho = rho + ins["amp"] * sum(
            float(a) * torch.sin(2 * math.pi * (float(k[0]) * x + float(k[1]) * y + float(k[2]) * z) + float(f))
            for a, k, f in zip(ins["a"], ins["k"], ins["phi"]))
    else:
        r2 = (x - ins["xc"][0]) ** 2 + (y - ins["xc"][1]) ** 2 + (z - ins["xc"][2]) ** 2
        rho, p = 1.0 + ins["amp"] * torch.exp(-r2 / ins["L"]), one
        vel = [v * one for v in ins["uinf"]]
    e = p / (gamma - 1) + 0.5 * rho * (vel[0] ** 2 + vel[1] ** 2 + vel[2] ** 2)
    return torch.stack([rho] + [rho * v for v in vel] + [e])


def _points(shape, nodes):
    """Coordinates of the nodes of every cell of the unit cube: three [cell][z][y][x]."""
    xi = torch.tensor(nodes, dtype=torch.float64, device=_device())
    ax = [(torch.arange(n, device=xi.device)[:, None] + xi[None, :]) / n for n in shape]
    z, y, x = ax[0][:, None, None, :, None, None], ax[1][None, :, None, None, :, None], ax[2][None, None, :, None, None, :]
    z, y, x = torch.broadcast_tensors(z, y, x)
    return [a.reshape((-1,) + a.shape[3:]) for a in (x, y, z)]


def _exact_dg(ins, order, shape, steps, gamma, cfl, ncp):
    ops = _Ops(order)
    nz, ny, nx = shape
    dx = (1.0 / nx, 1.0 / ny, 1.0 / nz)
    u = _start(ins, *_points(shape, ops.x), gamma).movedim(0, 1).contiguous()
    chunk = max(1, int(2.5e8 / (V * ops.B ** 4)))
    t, dt = 0.0, _dg_dt(u, dx, gamma, cfl, ncp)
    for _ in range(steps):
        u = _dg_step(u, shape, dt, dx, ops, gamma, ncp, chunk)
        t, dt = t + dt, _dg_dt(u, dx, gamma, cfl, ncp)
    return dict(t=t, dt=dt, u=u.movedim(1, -1).reshape(-1).contiguous())


def _exact_cell(case, seed):
    ops, dx = _Ops(case["order"]), (0.125, 0.1, 0.1)
    xi = torch.tensor(ops.x, dtype=torch.float64, device=_device()) - 0.5
    z, y, x = torch.meshgrid(0.45 + dx[2] * xi, 0.55 + dx[1] * xi, 0.5 + dx[0] * xi, indexing="ij")
    u = _start(_inputs(case, seed), x, y, z, GAMMA).unsqueeze(0)
    dt = _dg_dt(u, dx, GAMMA, CFL, False)
    qh, fh, q = _predict(u, dt, dx, ops, GAMMA, False)
    w = ops.w
    w3 = w[:, None, None] * w[None, :, None] * w[None, None, :]
    w2 = w[:, None] * w[None, :]
    dudt = torch.zeros_like(u)
    bq, bf, flux = [], [], []
    for d in range(3):
        (q0, q1), (f0, f1) = _faces(qh, d, ops), _faces(fh[d], d, ops)
        f = _riemann(q1, q0, f1, f0, d, w, GAMMA, False)[0]
        bq, bf, flux = bq + [q0, q1], bf + [f0, f1], flux + [f, f]
        dudt += (_contract(fh[d], ops.K.T.contiguous(), 4 - d)
                 - f.unsqueeze(4 - d) * _along(ops.right - ops.left, 4 - d, 5)) / _along(w, 4 - d, 5) / dx[d]
    face = lambda fs: torch.cat([f[0].movedim(0, -1).reshape(-1) for f in fs])  # noqa: E731
    new = u + dt * dudt
    nodes = lambda a: a[0].movedim(0, -1).reshape(-1)  # noqa: E731
    # the averaged fluxes in the layouts [z][y][x], [z][x][y], [y][x][z], then the (zero) source
    lf = [nodes(fh[0]), nodes(fh[1].permute(0, 1, 2, 4, 3)), nodes(fh[2].permute(0, 1, 3, 4, 2))]
    return dict(lQi=q[0].permute(2, 3, 4, 1, 0).reshape(-1), lQhi=nodes(qh),
                lFhi=torch.cat(lf + [torch.zeros_like(lf[0])]), lQhbnd=face(bq), lFhbnd=face(bf),
                flux=face(flux).reshape(6, -1), lduh=nodes(dudt * w3), luh=nodes(new), dt=_dg_dt(new, dx, GAMMA, CFL, False))


def _exact_fv(case, seed):
    """Both schemes on the whole periodic grid.  The half-step evolution of
    MUSCL-Hancock ends at a patch's own cells: across a patch boundary the
    neighbour's face state enters unevolved."""
    P, dim = case["patch"], case["dim"]
    shape = (case["nz"], case["ny"], case["nx"])
    n = [s * P for s in shape]
    dev = _device()
    ax = [(torch.arange(m, dtype=torch.float64, device=dev) + 0.5) / m for m in n]
    ins = _inputs(case, seed)
    if dim == 2:
        n[0] = 1
        ax[0] = torch.zeros(1, dtype=torch.float64, device=dev)
    z, y, x = torch.meshgrid(*ax, indexing="ij")
    u = _start(ins, x, y, z, GAMMA).unsqueeze(0)
    h = [1.0 / n[2], 1.0 / n[1], 1.0 / n[0]]

    def stable():
        return min(float((CFL / dim * h[d] / _speed(u, d, GAMMA)).min()) for d in range(dim))

    def rusanov(a, b, d):
        s = torch.maximum(_speed(a, d, GAMMA), _speed(b, d, GAMMA)).unsqueeze(1)
        return 0.5 * s * (a - b) + 0.5 * (_euler_flux(a, d, GAMMA) + _euler_flux(b, d, GAMMA))

    t, dt = 0.0, stable()
    for _ in range(case["steps"]):
        new = u.clone()
        if dim == 2:
            for d in range(2):
                f = rusanov(u, torch.roll(u, -1, 4 - d), d)
                new -= dt / h[d] * (f - torch.roll(f, 1, 4 - d))
        else:
            slopes, evolve = [], torch.zeros_like(u)
            for d in range(3):
                a, b = torch.roll(u, -1, 4 - d) - u, u - torch.roll(u, 1, 4 - d)
                s = 0.5 * torch.where(a * b < 0, torch.zeros_like(a), torch.where(a.abs() < b.abs(), a, b))
                evolve += 0.5 * dt / h[d] * (_euler_flux(u - s, d, GAMMA) - _euler_flux(u + s, d, GAMMA))
                slopes.append(s)
            for d in range(3):
                up, lo = u + slopes[d], u - slopes[d]
                i = _along(torch.arange(n[2 - d], device=dev) % P, 4 - d, 5)
                right = torch.roll(torch.where(i == 0, lo, lo + evolve), -1, 4 - d)
                left = torch.roll(torch.where(i == P - 1, up, up + evolve), 1, 4 - d)
                new -= dt / h[d] * (rusanov(up + evolve, right, d) - rusanov(left, lo + evolve, d))
        u = new
        t, dt = t + dt, stable()
    # [patch z][patch y][patch x][z][y][x][V]
    u = u[0].movedim(0, -1)
    if dim == 2:
        u = u[0].reshape(shape[1], P, shape[2], P, V).permute(0, 2, 1, 3, 4).reshape(-1, P, P, V)
    else:
        u = u.reshape(shape[0], P, shape[1], P, shape[2], P, V).permute(0, 2, 4, 1, 3, 5, 6).reshape(-1, P, P, P, V)
    return dict(t=t, dt=dt, u=u.contiguous())


def _exact_transfer(case, seed):
    """Prolongation evaluates the coarse polynomial at the children's nodes;
    restricting an exact embedding gives the coarse polynomial back."""
    ops, n = _Ops(case["order"]), case["n"] ** 3
    B = ops.B
    u = torch.tensor(1.0 + np.random.default_rng(seed).random(n * B ** 3 * V), device=_device())
    P = np.empty((3, B, B))
    for s in range(3):
        for k in range(B):
            for j in range(B):
                pts = (s + ops.x[j]) / 3.0
                P[s, k, j] = np.prod([(pts - ops.x[i]) / (ops.x[k] - ops.x[i]) for i in range(B) if i != k])
    P = torch.tensor(P, device=u.device)
    fine = torch.empty((n, 27, B, B, B, V), dtype=torch.float64, device=u.device)
    for s in range(27):
        a = u.reshape(n, B, B, B, V)
        for d, i in enumerate((s % 3, s // 3 % 3, s // 9)):
            a = _contract(a, P[i], 3 - d)
        fine[:, s] = a
    return dict(fine=fine.reshape(-1), back=u)


MOST_EXACT = 5e10  # values of the space-time iterate times steps: about 10 seconds


def exact(case, seed):
    kind = case["kind"]
    if kind == "cell":
        return _exact_cell(case, seed)
    if kind == "fv":
        return _exact_fv(case, seed)
    if kind == "transfer":
        return _exact_transfer(case, seed)
    if kind == "dg":
        cost = case["nx"] * case["ny"] * case["nz"] * case["steps"] * (case["order"] + 1) ** 4 * V
        if cost > MOST_EXACT:
            return None
        return _exact_dg(_inputs(case, seed), case["order"], (case["nz"], case["ny"], case["nx"]), case["steps"],
                         GAMMA, CFL, case["pde"] != "euler")
    if kind == "ensemble":
        out, cost = [], 0
        for m in _inputs(case, seed):
            one = m["cells"][0] ** 3 * case["steps"] * (m["order"] + 1) ** 4 * V
            if cost + one > MOST_EXACT:
                out.append(None)
                continue
            cost += one
            out.append(_exact_dg(m["ic"], m["order"], m["cells"], case["steps"], m["gamma"], CFL, False))
        return dict(t=None, dt=None, u=[None if r is None else r["u"] for r in out])
    # the adaptive limiting scheme is a state machine over statuses, patches
    # and hanging faces: no short formula for it
    return None
