"""Performance cases of the framework: what its users run, through its public
entry points, over the range of sizes, collision models, walls, storages and
launch paths they run it with.

The families (``kind`` of a case):

* ``lbm``     plain fused steps (``sim.LBM``): lid-driven cavities and channels in
  2D and 3D, FP32 and 16-bit storage, a chunk of steps per call as a program
  with on-line monitoring runs it.
* ``viv``     the 2D vortex-induced-vibration step with its histories (``sim.VIV2D``).
* ``sphere``  the 3D step past a fixed sphere (``sim.Sphere3D``).
* ``batch``   a parameter sweep advanced together (``sim.VIVBatch``).
* ``adjoint`` value and gradient of the VIV objective (``sim.VIVAdjoint``).
* ``ops_viv`` the VIV step composed by the user from the pure functions
  (``lbm``, ``ib``, ``dyn``), as the examples of the library compose it.
* ``ops3d``   a 3D cavity step composed from ``lbm3d`` and the field diagnostics of
  ``post`` a monitoring program evaluates after it.

``exact`` restates each family in float64 torch (no code of this repository).
"""

import math

import numpy as np
import torch

from vivsim_amd import dyn, ib, lbm, lbm3d, post, sim

DEV = "cuda"
GRIDS = ((256, 256), (512, 256), (512, 512), (1024, 512))   # the sweep's grids


def listed():
    return [
        # force-driven Poiseuille channel on a small grid: the shortest call, bound by latency
        dict(name="channel_small", kind="lbm", nx=96, ny=65, nz=0, walls="poiseuille", collision="mrt", storage="f32", steps=20),
        # the 256^2 lid-driven cavity of the documentation, a monitoring chunk of 100 steps
        dict(name="cavity_256", kind="lbm", nx=256, ny=256, nz=0, walls="cavity", collision="bgk", storage="f32", steps=100),
        # a mid-size cavity of odd sides in 16-bit storage with the entropic collision
        dict(name="cavity_kbc_f16s", kind="lbm", nx=1031, ny=777, nz=0, walls="cavity_bb", collision="kbc", storage="f16s", steps=50),
        # a long channel with velocity inlet, pressure outlet and solid walls, beyond the last-level cache
        dict(name="channel_large", kind="lbm", nx=4000, ny=2050, nz=0, walls="channel", collision="bgk", storage="f32", steps=20),
        # 3D lid-driven cavity, odd sides
        dict(name="cavity3d", kind="lbm", nx=121, ny=113, nz=127, walls="cavity", collision="mrt", storage="f32", steps=20),
        # the headline VIV step, one output chunk
        dict(name="viv_1024", kind="viv", nx=1024, ny=1024, D=40.0, markers=512, collision="mrt", forcing="guo", storage="f32", steps=50),
        # the same body in a grid beyond the last-level cache, 16-bit storage
        dict(name="viv_4096_f16s", kind="viv", nx=4096, ny=4096, D=40.0, markers=512, collision="mrt", forcing="guo", storage="f16s", steps=20),
        # 3D flow past a sphere
        dict(name="sphere", kind="sphere", nx=256, ny=128, nz=128, D=24.0, markers=4096, collision="bgk", forcing="edm", storage="f32", steps=20),
        # a sweep of 16 cases over the four grids
        dict(name="batch16", kind="batch", cases=16, storage="f32", steps=50),
        # one objective and gradient of a shape / stiffness optimisation
        dict(name="adjoint", kind="adjoint", nx=512, ny=256, D=32.0, markers=256, steps=150),
        # the step as a user of the pure functions writes it
        dict(name="ops_viv", kind="ops_viv", nx=512, ny=400, D=30.0, markers=120, steps=4),
        # 3D pure functions and diagnostics, odd sides
        dict(name="ops3d", kind="ops3d", nx=129, ny=97, nz=110, collision="mrt", steps=2),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same families and ranges."""
    kind = rng.choice(["lbm", "lbm", "lbm3", "viv", "viv", "sphere", "batch", "adjoint", "ops_viv", "ops3d"])
    if kind in ("lbm", "lbm3"):
        three = kind == "lbm3"
        collision = rng.choice(["bgk", "mrt", "kbc", "reg"])
        if three:
            nx, ny, nz = (_log(rng, 24, 160) for _ in range(3))
            walls = rng.choice(["cavity", "cavity_bb", "duct", "periodic"])
        else:
            nx, ny, nz = _log(rng, 40, 4000), _log(rng, 40, 2050), 0
            walls = rng.choice(["cavity", "cavity_bb", "channel", "poiseuille", "periodic"])
        storage = rng.choice(["f32", "f32", "f16s", "bf16s", "e3m12s"])
        most = int(1.6e8 if not three else 4.5e7) // (nx * ny * max(nz, 1))
        return dict(kind="lbm", nx=nx, ny=ny, nz=nz, walls=walls, collision=collision, storage=storage,
                    steps=max(1, min(_log(rng, 2, 150), most)))
    if kind == "viv":
        D = rng.choice([16.0, 20.0, 32.0, 40.0, 48.0])
        nx, ny = _log(rng, 180, 4096), _log(rng, 180, 4096)
        most = int(3.2e8) // (nx * ny)
        return dict(kind="viv", nx=nx, ny=ny, D=D, markers=int(D * rng.choice([4, 8, 12.8])),
                    collision=rng.choice(["mrt", "bgk", "kbc"]), forcing=rng.choice(["guo", "edm"]),
                    storage=rng.choice(["f32", "f32", "f16s", "e3m12s"]), steps=max(2, min(_log(rng, 5, 100), most)))
    if kind == "sphere":
        D = float(rng.choice([12, 16, 24]))
        nx, ny, nz = _log(rng, 64, 256), _log(rng, 48, 140), _log(rng, 48, 140)
        return dict(kind="sphere", nx=nx, ny=ny, nz=nz, D=D, markers=int(D * D * rng.uniform(4, 7.5)),
                    collision=rng.choice(["bgk", "mrt"]), forcing=rng.choice(["edm", "guo"]),
                    storage=rng.choice(["f32", "f16s"]), steps=_log(rng, 4, 20))
    if kind == "batch":
        return dict(kind="batch", cases=rng.randint(2, 24), storage=rng.choice(["f32", "f16s"]), steps=_log(rng, 10, 50))
    if kind == "adjoint":
        D = float(rng.choice([16, 24, 32]))
        return dict(kind="adjoint", nx=_log(rng, 128, 512), ny=_log(rng, 96, 256), D=D, markers=int(D * 8), steps=_log(rng, 100, 150))
    if kind == "ops_viv":
        D = float(rng.choice([16, 24, 30, 40]))
        return dict(kind="ops_viv", nx=_log(rng, 128, 1200), ny=_log(rng, 100, 1100), D=D, markers=int(D * 4), steps=rng.randint(1, 6))
    nx, ny, nz = (_log(rng, 32, 140) for _ in range(3))
    return dict(kind="ops3d", nx=nx, ny=ny, nz=nz, collision=rng.choice(["bgk", "mrt", "kbc", "reg"]), steps=rng.randint(1, 3))


# ---------------------------------------------------------------- inputs

U0 = 0.05


def _wall_list(name, three):
    """Ordered wall lists of the cavity and channel programs."""
    lid = dict(ux_wall=U0)
    sides = ("left", "right", "bottom", "top") + (("back", "front") if three else ())
    if name == "cavity":
        return [dict(kind="nee", mode="plain", loc=s, **(lid if s == "top" else {})) for s in sides]
    if name == "cavity_bb":
        return [dict(kind="bb", loc=s, **(lid if s == "top" else {})) for s in sides]
    if name == "channel":
        return [dict(kind="nebb", mode="velocity", loc="left", ux_wall=U0), dict(kind="nebb", mode="pressure", loc="right", rho_wall=1.0),
                dict(kind="bb", loc="bottom"), dict(kind="bb", loc="top")]
    if name == "duct":
        return [dict(kind="eq", mode="plain", loc="left", ux_wall=U0), dict(kind="nee", mode="pressure", loc="right", rho_wall=1.0),
                dict(kind="bb", loc="bottom"), dict(kind="bb", loc="top")]
    if name == "poiseuille":
        return [dict(kind="bb", loc="bottom"), dict(kind="bb", loc="top")]
    return []


def _forced(c):
    return c["walls"] in ("poiseuille", "periodic")


def _omega(c):
    """Relaxation rate of the plain flows (nu = 0.02)."""
    return 1 / (3 * 0.02 + 0.5)


def _uniform(seed, shape, lo, hi, dtype=torch.float32):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return torch.rand(shape, generator=g, device=DEV, dtype=dtype) * (hi - lo) + lo


def _start_field(seed, shape, u0):
    """Equilibrium of a flow at u0 with 1 % velocity and density perturbations: the caller's f[Q, *shape]."""
    d = len(shape)
    u = _uniform(seed, (d,) + tuple(shape), -0.01 * U0, 0.01 * U0)
    u[0] += u0
    rho = _uniform(seed + 1, tuple(shape), 0.999, 1.001)
    return _equilibrium(rho, u).contiguous()


def _viv_case(c, seed=0, **kw):
    # the adjoint's body sits near the inlet, whose velocity it differentiates
    cx = c["D"] / 2 + 30 if c["kind"] == "adjoint" else c["nx"] // 4 + int(c["D"]) // 2 + 8
    return sim.VIVCase(nx=c["nx"], ny=c["ny"], D=c["D"], cx=float(cx), cy=float(c["ny"] // 2),
                       n_markers=c["markers"], U0=U0, collision=c.get("collision", "mrt"), forcing=c.get("forcing", "guo"), seed=seed, **kw)


def _batch_cases(c, seed):
    """KBC + EDM cases as a sweep draws them: grid, reduced velocity, Reynolds number, mass ratio."""
    rng = np.random.default_rng(seed)
    out = []
    for k in range(c["cases"]):
        nx, ny = GRIDS[k % len(GRIDS)]
        D = ny / 8
        out.append(sim.VIVCase(nx=nx, ny=ny, D=D, cx=nx / 4, cy=ny / 2, n_markers=int(round(np.pi * D / 0.75)), Ur=float(rng.uniform(3, 8)),
                               Re=float(rng.uniform(100, 1000)), mass_ratio=float(rng.uniform(1, 10)), collision="kbc", forcing="edm", n_iter=3))
    return out


def _sphere_case(c):
    return sim.SphereCase(nx=c["nx"], ny=c["ny"], nz=c["nz"], D=c["D"], cx=float(c["nx"] // 4 + 6), cy=float(c["ny"] // 2), cz=float(c["nz"] // 2),
                          n_markers=c["markers"], U0=U0, collision=c["collision"], forcing=c["forcing"])


def prepare(case, seed):
    c, k = case, case["kind"]
    torch.cuda.set_device(0)
    s = dict(case=c)
    if k == "lbm":
        shape = (c["nx"], c["ny"]) + ((c["nz"],) if c["nz"] else ())
        kw = dict(forcing="guo", g_uniform=(1e-6,) + (0.0,) * (len(shape) - 1)) if _forced(c) else {}
        s["solver"] = sim.LBM(shape, _omega(c), collision=c["collision"], walls=_wall_list(c["walls"], len(shape) == 3), storage=c["storage"], **kw)
        s["f"] = _start_field(seed, shape, U0 if c["walls"] in ("channel", "duct") else 0.0)
        s["out"] = torch.empty_like(s["f"])
    elif k == "viv":
        s["solver"] = sim.VIV2D(_viv_case(c), storage=c["storage"])
        s["solver"].set_body(v=(0.0, 1e-3 * U0))
        s["f"] = _start_field(seed, (c["nx"], c["ny"]), U0)
        s["out"] = torch.empty_like(s["f"])
    elif k == "sphere":
        s["solver"] = sim.Sphere3D(_sphere_case(c), storage=c["storage"])
        s["f"] = _start_field(seed, (c["nx"], c["ny"], c["nz"]), U0)
        s["out"] = torch.empty_like(s["f"])
    elif k == "batch":
        cases = _batch_cases(c, seed)
        s["solver"] = b = sim.VIVBatch(cases, storage=c["storage"])
        b.set_bodies(v=(0.0, 5e-5))
        s["f"] = torch.zeros(b.total, device=DEV)
        for j, vc in enumerate(cases):
            b.view(s["f"], j).copy_(_start_field(seed + 2 * j, (vc.nx, vc.ny), U0))
        s["out"] = torch.empty_like(s["f"])
    elif k == "adjoint":
        s["solver"] = sim.VIVAdjoint(_viv_case(c, seed=seed, Re=150.0), c["steps"], v0=(0.0, 1e-3 * U0))
        s["delta"] = _uniform(seed, (c["markers"],), -0.1, 0.1, torch.float64)
    elif k == "ops_viv":
        vc = _viv_case(c)
        mx, my = vc.markers()
        f64 = dict(dtype=torch.float64, device=DEV)
        s.update(vc=vc, f=_start_field(seed, (c["nx"], c["ny"]), U0), mx=torch.as_tensor(mx, dtype=torch.float32, device=DEV),
                 my=torch.as_tensor(my, dtype=torch.float32, device=DEV), a=torch.zeros(2, **f64),
                 v=torch.tensor([0.0, 1e-3 * U0], **f64), d=torch.zeros(2, **f64), op=lbm.get_mrt_collision_operator(vc.omega),
                 fop=lbm.get_mrt_forcing_operator(vc.omega))
    else:
        s["f"] = _start_field(seed, (c["nx"], c["ny"], c["nz"]), 0.0)
        s["op"] = lbm3d.get_mrt_collision_operator(_omega(c))
    return s


# ---------------------------------------------------------------- one pass

def _ops_viv_step(s):
    """One VIV step from the pure functions (window fixed in the grid: the body moves by far less than its margin)."""
    vc = s["vc"]
    S, x0, y0 = vc.ib_size, vc.ib_x0, vc.ib_y0
    f, d, v, a = s["f"], s["d"], s["v"], s["a"]
    rho, u = lbm.get_macroscopic(f)
    mx, my = dyn.get_markers_coords_2dof(s["mx"], s["my"], d)
    W, idx = ib.get_ib_stencil(mx - x0, my - y0, S)
    g_win, h_m = ib.multi_direct_forcing(u[:, x0:x0 + S, y0:y0 + S], W, idx, v.to(torch.float32).expand(vc.n_markers, 2), vc.ds, vc.n_iter)
    h = dyn.get_force_to_obj(h_m) + a * vc.area
    s["a"], s["v"], s["d"] = dyn.newmark_2dof(a, v, d, h, vc.mass, vc.stiffness, vc.damping)
    g = torch.zeros_like(u)
    g[:, x0:x0 + S, y0:y0 + S] = g_win
    u = u + lbm.get_velocity_correction(g, rho)
    feq = lbm.get_equilibrium(rho, u)
    f = lbm.collision_mrt(f, feq, s["op"])
    f = lbm.forcing_guo_mrt(f, g, u, s["fop"])
    f = lbm.streaming(f)
    f = lbm.boundary_equilibrium(f, "left", ux_wall=U0)
    s["f"] = lbm.boundary_pressure_nee(f, "right", rho_wall=1.0)
    return h_m


def run(state):
    s, c = state, state["case"]
    k = c["kind"]
    if k == "lbm":
        s["f"], s["out"] = s["solver"].run(s["f"], c["steps"], out=s["out"]), s["f"]
        return s["f"]
    if k == "viv":
        f, d, h = s["solver"].run(s["f"], c["steps"], out=s["out"])
        s["f"], s["out"] = f, s["f"]
        return f, d, h
    if k == "sphere":
        f, h = s["solver"].run(s["f"], c["steps"], out=s["out"])
        s["f"], s["out"] = f, s["f"]
        return f, h
    if k == "batch":
        f = s["solver"].run(s["f"], c["steps"], out=s["out"])
        s["f"], s["out"] = f, s["f"]
        return f
    if k == "adjoint":
        vc = s["solver"].case
        return s["solver"].evaluate(s["delta"], vc.stiffness, vc.U0)
    if k == "ops_viv":
        for _ in range(c["steps"]):
            h_m = _ops_viv_step(s)
        return s["f"], s["d"], s["v"], h_m
    om = _omega(c)
    f = s["f"]
    for _ in range(c["steps"]):
        rho, u = lbm3d.get_macroscopic(f)
        feq = lbm3d.get_equilibrium(rho, u)
        col = c["collision"]
        if col == "mrt":
            f = lbm3d.collision_mrt(f, feq, s["op"])
        else:
            f = dict(bgk=lbm3d.collision_bgk, kbc=lbm3d.collision_kbc, reg=lbm3d.collision_reg)[col](f, feq, om)
        f = lbm3d.streaming(f)
        for loc in ("left", "right", "bottom", "back", "front"):
            f = lbm3d.boundary_nee(f, loc)
        f = lbm3d.boundary_nee(f, "top", ux_wall=U0)
    s["f"] = f
    rho, u = lbm3d.get_macroscopic(f)
    return f, rho, u, post.vorticity(u), post.q_criterion(u)


# ---------------------------------------------------------------- work

# operations of one cell update (moments, equilibrium, relaxation; a multiply-add counts two)
FLOPS = {("bgk", 2): 130, ("mrt", 2): 190, ("kbc", 2): 240, ("reg", 2): 170, ("bgk", 3): 300, ("mrt", 3): 620, ("kbc", 3): 700, ("reg", 3): 500}


def work(case):
    """One call's inputs read once and its outputs written once, and the arithmetic of its steps."""
    c, k = case, case["kind"]
    if k == "batch":
        cells, q, col = sum(GRIDS[j % 4][0] * GRIDS[j % 4][1] for j in range(c["cases"])), 9, ("kbc", 2)
    else:
        three = bool(c.get("nz"))
        cells, q = c["nx"] * c["ny"] * (c["nz"] if three else 1), 19 if three else 9
        col = (c.get("collision", "mrt"), 3 if three else 2)
    flops = cells * c["steps"] * FLOPS[col]
    bytes_ = 2 * 4 * q * cells
    if k == "adjoint":
        # the initial field once; a reverse step costs about twice a forward one, which runs twice
        return dict(bytes=4 * q * cells, flops=4 * flops)
    if k == "ops_viv":
        # per step, by function: macroscopic, correction, equilibrium, collision, forcing, streaming, two walls
        return dict(bytes=4 * cells * c["steps"] * (12 + 7 + 12 + 27 + 22 + 18 + 2 * 18), flops=flops)
    if k == "ops3d":
        per = 23 + 23 + 57 + 38 + 6 * 38
        return dict(bytes=4 * cells * (c["steps"] * per + 23 + 6 + 4), flops=flops)
    return dict(bytes=bytes_, flops=flops)


# ---------------------------------------------------------------- the same in float64 torch

C2 = [(0, 0), (1, 0), (0, 1), (-1, 0), (0, -1), (1, 1), (-1, 1), (-1, -1), (1, -1)]
C3 = [(0, 0, 0), (1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1), (1, 1, 0), (-1, 1, 0), (1, -1, 0), (-1, -1, 0),
      (1, 0, 1), (-1, 0, 1), (1, 0, -1), (-1, 0, -1), (0, 1, 1), (0, -1, 1), (0, 1, -1), (0, -1, -1)]
FACES = dict(left=(0, 1), right=(0, -1), bottom=(1, 1), top=(1, -1), back=(2, 1), front=(2, -1))   # axis, inward sign
IN2 = dict(left=(1, 5, 8), right=(3, 7, 6), bottom=(2, 5, 6), top=(4, 7, 8))
OUT2 = dict(left=(3, 7, 6), right=(1, 5, 8), bottom=(4, 7, 8), top=(2, 5, 6))


def _lattice(d):
    cs = C2 if d == 2 else C3
    zero, one, two = (4 / 9, 1 / 9, 1 / 36) if d == 2 else (1 / 3, 1 / 18, 1 / 36)
    return cs, [(zero, one, two)[sum(map(abs, c))] for c in cs]


def _dot(c, u):
    """c . u for an integer direction (zero components skipped)."""
    r = None
    for a, ca in enumerate(c):
        if ca:
            t = u[a] if ca > 0 else -u[a]
            r = t if r is None else r + t
    return torch.zeros_like(u[0]) if r is None else r


def _equilibrium(rho, u):
    cs, w = _lattice(u.shape[0])
    base = 1 - 1.5 * (u * u).sum(0)
    out = []
    for c, wi in zip(cs, w):
        cu = _dot(c, u)
        out.append(rho * wi * (base + 3 * cu + 4.5 * cu * cu))
    return torch.stack(out)


def _macroscopic(f):
    cs, _ = _lattice(2 if f.shape[0] == 9 else 3)
    rho = f.sum(0)
    u = [sum(f[i] * float(c[a]) for i, c in enumerate(cs) if c[a]) / rho for a in range(len(cs[0]))]
    return rho, torch.stack(u)


def _guo(g, u):
    cs, w = _lattice(u.shape[0])
    gu = (g * u).sum(0)
    return torch.stack([wi * (3 * (_dot(c, g) - gu) + 9 * _dot(c, g) * _dot(c, u)) for c, wi in zip(cs, w)])


def _moments(d):
    """Rows of the moment basis and the index of the rates that follow omega."""
    if d == 2:
        return np.array([[1] * 9, [-4, -1, -1, -1, -1, 2, 2, 2, 2], [4, -2, -2, -2, -2, 1, 1, 1, 1], [0, 1, 0, -1, 0, 1, -1, -1, 1],
                         [0, -2, 0, 2, 0, 1, -1, -1, 1], [0, 0, 1, 0, -1, 1, 1, -1, -1], [0, 0, -2, 0, 2, 1, 1, -1, -1],
                         [0, 1, -1, 1, -1, 0, 0, 0, 0], [0, 0, 0, 0, 0, 1, -1, 1, -1]], dtype=np.float64)
    x, y, z = np.array(C3, dtype=np.float64).T
    q = x * x + y * y + z * z
    return np.array([np.ones(19), x, y, z, q, 3 * x * x - q, y * y - z * z, x * y, x * z, y * z, x * x * y, x * x * z, x * y * y, y * y * z,
                     x * z * z, y * z * z, x * x * y * y, x * x * z * z, y * y * z * z])


def _mrt(d, om):
    """Collision and forcing operators M^-1 S M and M^-1 (1 - S / 2) M."""
    m = _moments(d)
    rates = [0, 1.4, 1.4, 0, 1.2, 0, 1.2, om, om] if d == 2 else [0, 0, 0, 0, 1.1] + [om] * 5 + [1.2] * 6 + [1.4] * 3
    inv = np.linalg.inv(m)
    s = np.diag(rates)
    return tuple(torch.tensor(x, device=DEV) for x in (inv @ s @ m, inv @ (np.eye(len(rates)) - s / 2) @ m))


def _apply(op, x):
    return (op @ x.reshape(x.shape[0], -1)).reshape(x.shape)


def _project(x):
    """Second-order Hermite projection of a non-equilibrium part."""
    cs, w = _lattice(2 if x.shape[0] == 9 else 3)
    c = np.array(cs, dtype=np.float64)
    d = c.shape[1]
    h = np.einsum("qa,qb->qab", c, c) - np.eye(d) / 3
    return _apply(torch.tensor(4.5 * np.array(w)[:, None] * np.einsum("qab,ra,rb->qr", h, c, c), device=DEV), x)


def _shear2(x):
    """Shear part of the 2D entropic collision."""
    n, p = (x[1] - x[2] + x[3] - x[4]) / 4, (x[5] - x[6] + x[7] - x[8]) / 4
    return torch.stack([torch.zeros_like(n), n, -n, n, -n, p, -p, p, -p])


def _collide(f, rho, u, om, collision, forcing=None, g=None):
    if forcing == "guo":
        u = u + 0.5 * g / rho
    feq = _equilibrium(rho, u)
    d = u.shape[0]
    if collision == "bgk":
        out = f + om * (feq - f)
    elif collision == "mrt":
        op, fop = _mrt(d, om)
        out = f + _apply(op, feq - f)
    elif collision == "reg":
        out = feq + (1 - om) * _project(f - feq)
    else:
        neq = f - feq
        s = _shear2(neq) if d == 2 else _project(neq)
        h = neq - s
        gam = 1 / om - (1 - 1 / om) * (h * s / feq).sum(0) / ((h * h / feq).sum(0) + 1e-20)
        out = f - om * (s + gam * h)
    if forcing is None:
        return out
    F = _guo(g, u)
    if forcing == "edm":
        return out + F
    return out + (_apply(fop, F) if collision == "mrt" else (1 - 0.5 * om) * F)


def _stream(f):
    cs, _ = _lattice(2 if f.shape[0] == 9 else 3)
    return torch.stack([torch.roll(f[i], shifts=c, dims=tuple(range(len(c)))) for i, c in enumerate(cs)])


def _line(f, loc, layer):
    axis, sign = FACES[loc]
    return f.select(1 + axis, layer if sign > 0 else f.shape[1 + axis] - 1 - layer)


def _walls(f, pre, walls):
    """The ordered walls on a streamed field (a new tensor, differentiable)."""
    d = f.dim() - 1
    cs, w = _lattice(d)
    for wl in walls:
        loc, kind, mode = wl["loc"], wl["kind"], wl.get("mode", "plain")
        axis, sign = FACES[loc]
        x, nb = _line(f, loc, 0), _line(f, loc, 1)
        u = torch.stack([torch.as_tensor(wl.get(n, 0.0), dtype=f.dtype, device=f.device).expand(x.shape[1:]) for n in ("ux_wall", "uy_wall", "uz_wall")[:d]])
        rho = torch.full_like(x[0], wl.get("rho_wall", 1.0))
        cn = [c[axis] * sign for c in cs]
        num = sum(x[i] * (1.0 if n == 0 else 2.0) for i, n in enumerate(cn) if n <= 0)
        if mode == "velocity":
            rho = num / (1 - sign * u[axis])
        elif mode == "pressure":
            _, un = _line_macro(nb, cs)
            u = torch.stack([sign * (1 - num / rho) if a == axis else un[a] for a in range(d)])
        if kind in ("eq", "nee"):
            new = _line_eq(rho, u, cs, w)
            if kind == "nee":
                rn, un = _line_macro(nb, cs)
                new = new + nb - _line_eq(rn, un, cs, w)
        else:
            new = list(x.unbind(0))
            p = _line(pre, loc, 0)
            inn = IN2[loc] if d == 2 else [i for i, n in enumerate(cn) if n > 0]
            if kind == "bb" and d == 2:
                un, ut = sign * u[axis], sign * u[1 - axis]
                for i, o, add in zip(inn, OUT2[loc], (2 / 3 * un, (un + ut) / 6, (un - ut) / 6)):
                    new[i] = p[o] + add
            elif kind == "bb":
                out = [i for i, n in enumerate(cn) if n < 0]
                for i, o in zip(inn, out):
                    new[i] = p[o] + 6 * w[i] * p.sum(0) * _dot(cs[i], u)
            else:   # Zou / He (2D)
                un, ut = sign * u[axis], sign * u[1 - axis]
                t = (2, 4) if axis == 0 else (1, 3)
                sh = 0.5 * (x[t[0]] - x[t[1]]) * sign
                for i, o, add in zip(inn, OUT2[loc], (2 / 3 * un * rho, -sh + un * rho / 6 + ut * rho / 2, sh + un * rho / 6 - ut * rho / 2)):
                    new[i] = x[o] + add
            new = torch.stack(new)
        n = f.shape[1 + axis]
        new = new.unsqueeze(1 + axis)
        f = torch.cat([new, f.narrow(1 + axis, 1, n - 1)] if sign > 0 else [f.narrow(1 + axis, 0, n - 1), new], dim=1 + axis)
    return f


def _line_macro(x, cs):
    rho = x.sum(0)
    return rho, torch.stack([sum(x[i] * float(c[a]) for i, c in enumerate(cs) if c[a]) / rho for a in range(len(cs[0]))])


def _line_eq(rho, u, cs, w):
    base = 1 - 1.5 * (u * u).sum(0)
    return torch.stack([rho * wi * (base + 3 * _dot(c, u) + 4.5 * _dot(c, u) ** 2) for c, wi in zip(cs, w)])


def _phi(r):
    """Peskin's 4-point kernel."""
    a = r.abs()
    inner = (3 - 2 * a + torch.sqrt((1 + 4 * a - 4 * a * a).clamp(min=0))) / 8
    outer = (5 - 2 * a - torch.sqrt((-7 + 12 * a - 4 * a * a).clamp(min=0))) / 8
    return torch.where(a > 2, torch.zeros_like(a), torch.where(a < 1, inner, outer))


def _stencil(x, size):
    """Weights and flat indices of markers x[M, d] in a cubic window."""
    off = torch.arange(-1, 3, device=x.device)
    w, idx = None, None
    for a in range(x.shape[1]):
        s = torch.floor(x[:, a].detach()).long()[:, None] + off
        p = _phi(s - x[:, a:a + 1])
        w = p if w is None else (w[:, :, None] * p[:, None, :]).flatten(1)
        idx = s if idx is None else (idx[:, :, None] * size + s[:, None, :]).flatten(1)
    return w, idx


def _mdf(u, w, idx, target, ds, n_iter):
    """Multi-direct forcing in a window: force grid and total marker forces."""
    flat = u.reshape(u.shape[0], -1)

    def interp(g):
        return (w[None] * g[:, idx]).sum(2).t()

    def spread(F):
        v = (F.t()[:, :, None] * w[None]).flatten(1)
        return torch.zeros_like(flat).index_add(1, idx.reshape(-1), v)

    ub, F = interp(flat), torch.zeros_like(target)
    for _ in range(n_iter):
        dF = (target - ub) * (2 * ds)
        F = F + dF
        ub = ub + interp(0.5 * spread(dF))
    return spread(F).reshape(u.shape), F


def _place(g, start, shape):
    pad = []
    for a in reversed(range(len(shape))):
        pad += [start[a], shape[a] - start[a] - g.shape[1 + a]]
    return torch.nn.functional.pad(g, pad)


def _viv_exact(vc, f, steps, v0, delta=None, stiffness=None, u_in=None, fixed=False):
    """steps of the VIV flow in float64: f, body, histories and the last marker forces."""
    S = vc.ib_size
    th = 2 * np.pi * torch.arange(vc.n_markers, device=DEV, dtype=torch.float64) / vc.n_markers
    R = 0.5 * vc.D + (0.0 if delta is None else delta)
    mx, my = vc.cx + R * torch.cos(th), vc.cy + R * torch.sin(th)
    K = vc.stiffness if stiffness is None else stiffness
    z = torch.zeros(2, dtype=torch.float64, device=DEV)
    d, v, a = z, torch.tensor(v0, dtype=torch.float64, device=DEV), z
    mask = torch.tensor([1.0, 1.0] if fixed else [float(x) for x in vc.dof], dtype=torch.float64, device=DEV)
    walls = [dict(kind="eq", loc="left", ux_wall=U0 if u_in is None else u_in), dict(kind="nee", mode="pressure", loc="right")]
    dh, hh, hm = [], [], None
    for _ in range(steps):
        rho, u = _macroscopic(f)
        x0 = vc.ib_x0 if fixed else int(math.trunc(vc.ib_x0 + float(d[0].detach())))
        y0 = vc.ib_y0 if fixed else int(math.trunc(vc.ib_y0 + float(d[1].detach())))
        w, idx = _stencil(torch.stack([mx + d[0] - x0, my + d[1] - y0], 1), S)
        gw, F = _mdf(u[:, x0:x0 + S, y0:y0 + S], w, idx, v[None].expand(vc.n_markers, 2), vc.ds, vc.n_iter)
        hm = -F
        h = hm.sum(0) + a * vc.area
        v1, d1 = v + 0.5 * a, d + v + 0.25 * a
        an = (h - vc.damping * v1 - K * d1) / (vc.mass + 0.5 * vc.damping + 0.25 * K)
        a, v, d = an * mask, (0.5 * an + v1) * mask, (0.25 * an + d1) * mask
        g = _place(gw, (x0, y0), u.shape[1:])
        post_f = _collide(f, rho, u, vc.omega, vc.collision, vc.forcing, g)
        f = _walls(_stream(post_f), post_f, walls)
        dh.append(d)
        hh.append(h)
    return f, d, v, torch.stack(dh), torch.stack(hh), hm


def _grad(x, axis):
    inner = (x.narrow(axis, 2, x.shape[axis] - 2) - x.narrow(axis, 0, x.shape[axis] - 2)) / 2
    lo = x.narrow(axis, 1, 1) - x.narrow(axis, 0, 1)
    n = x.shape[axis]
    return torch.cat([lo, inner, x.narrow(axis, n - 1, 1) - x.narrow(axis, n - 2, 1)], axis)


def exact(case, seed):
    c, k = case, case["kind"]
    v0 = [0.0, 1e-3 * U0]
    if k == "lbm":
        shape = (c["nx"], c["ny"]) + ((c["nz"],) if c["nz"] else ())
        f = _start_field(seed, shape, U0 if c["walls"] in ("channel", "duct") else 0.0).double()
        walls = _wall_list(c["walls"], len(shape) == 3)
        g = None
        if _forced(c):
            g = torch.zeros((len(shape),) + (1,) * len(shape), dtype=torch.float64, device=DEV)
            g[0] = 1e-6
            g = g.expand((len(shape),) + shape)
        for _ in range(c["steps"]):
            rho, u = _macroscopic(f)
            p = _collide(f, rho, u, _omega(c), c["collision"], "guo" if g is not None else None, g)
            f = _walls(_stream(p), p, walls)
        return f
    if k == "viv":
        f, _, _, d, h, _ = _viv_exact(_viv_case(c), _start_field(seed, (c["nx"], c["ny"]), U0).double(), c["steps"], v0)
        return f, d, h
    if k == "batch":
        out, at = [], 0
        for j, vc in enumerate(_batch_cases(c, seed)):
            f = _viv_exact(vc, _start_field(seed + 2 * j, (vc.nx, vc.ny), U0).double(), c["steps"], [0.0, 5e-5])[0]
            out.append(f.reshape(-1))
            at += f.numel()   # every grid of the sweep is a multiple of 64 populations: no gaps
        return torch.cat(out)
    if k == "sphere":
        sc = _sphere_case(c)
        S, o = sc.ib_size, sc.ib_origin
        f = _start_field(seed, (c["nx"], c["ny"], c["nz"]), U0).double()
        rel = torch.as_tensor(sc.markers() - np.array(o, dtype=np.float64), device=DEV)
        w, idx = _stencil(rel, S)
        target = torch.zeros((c["markers"], 3), dtype=torch.float64, device=DEV)
        walls = [dict(kind="eq", loc="left", ux_wall=U0), dict(kind="nee", mode="pressure", loc="right")]
        hist = []
        for _ in range(c["steps"]):
            rho, u = _macroscopic(f)
            gw, F = _mdf(u[:, o[0]:o[0] + S, o[1]:o[1] + S, o[2]:o[2] + S], w, idx, target, sc.ds, sc.n_iter)
            hist.append(-F.sum(0))
            p = _collide(f, rho, u, sc.omega, c["collision"], c["forcing"], _place(gw, o, u.shape[1:]))
            f = _walls(_stream(p), p, walls)
        return f, torch.stack(hist)
    if k == "adjoint":
        vc = _viv_case(c, seed=seed, Re=150.0)
        u = torch.as_tensor(vc.initial_u(), dtype=torch.float32, device=DEV)
        f = _equilibrium(torch.ones_like(u[0]), u).double()
        delta = _uniform(seed, (c["markers"],), -0.1, 0.1, torch.float64).requires_grad_()
        K = torch.tensor(vc.stiffness, dtype=torch.float64, device=DEV, requires_grad=True)
        ui = torch.tensor(U0, dtype=torch.float64, device=DEV, requires_grad=True)
        dh = _viv_exact(vc, f, c["steps"], v0, delta, K, ui)[3]
        J = (dh[:, 1] ** 2).mean()
        gd, gk, gu = torch.autograd.grad(J, (delta, K, ui))
        return float(J.detach()), gd, float(gk), float(gu)
    if k == "ops_viv":
        f, d, v, _, _, hm = _viv_exact(_viv_case(c), _start_field(seed, (c["nx"], c["ny"]), U0).double(), c["steps"], v0, fixed=True)
        return f, d, v, hm
    om = _omega(c)
    f = _start_field(seed, (c["nx"], c["ny"], c["nz"]), 0.0).double()
    walls = [dict(kind="nee", loc=s) for s in ("left", "right", "bottom", "back", "front")] + [dict(kind="nee", loc="top", ux_wall=U0)]
    for _ in range(c["steps"]):
        rho, u = _macroscopic(f)
        p = _collide(f, rho, u, om, c["collision"])
        f = _walls(_stream(p), p, walls)
    rho, u = _macroscopic(f)
    G = [[_grad(u[i], j) for j in range(3)] for i in range(3)]
    vort = torch.stack([G[2][1] - G[1][2], G[0][2] - G[2][0], G[1][0] - G[0][1]])
    q = -0.5 * sum(G[i][j] * G[j][i] for i in range(3) for j in range(3))
    return f, rho, u, vort, q
