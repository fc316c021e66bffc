"""What this framework is run for, as cases that can be timed and compared.

A case is a dict of plain values.  ``prepare(case, seed)`` makes what a program holds before the call (program
handle, device fields, ensemble or adjoint handle), ``run(state)`` is one pass through the public entry points,
``work(case)`` the bytes and operations the pass cannot do without, and ``exact(case, seed)`` the same results in
64 bits from dense one-dimensional operators, without the library.

Kinds of case:

* ``uniform``   -- periodic box, uniform velocity and density, whole RK steps through ``Program.step``
* ``lists``     -- whole RK steps through the reference's kernel lists (``Program.run``): bounded or periodic grids,
                   velocity fields (static or time-dependent), with or without the Hall term, SATs, dissipation
* ``ensemble``  -- many periodic boxes advanced together (``Ensemble.step``)
* ``adjoint``   -- a solve and its gradient (``hall_solve`` under torch.autograd)
* ``clean``     -- divergence cleaning by CG (``Program.clean_div_cg``)
* ``series``    -- a driver run with integrals over time and cleaning after every step (host arrays in and out)
* ``diagnose``  -- energy, divergence norm and error norm of a field (``Program.diagnostics``)
"""
import math

import numpy as np
import torch

TWO_PI = 2 * math.pi
REAL = {"f64": "double", "f32": "float"}
ORDER = {"2ndOrder": 2, "4thOrder": 4, "6thOrder": 6, "2ndOrderExtended": 2, "4thOrderExtended": 4, "6thOrderExtended": 6}
STAGES = {"SSPRK33": 3, "SSPRK104": 10, "KennedyCarpenterLewis2R54C": 5, "CalvoFrancoRandez2R64": 6,
          "CarpenterKennedy2N54": 5, "ToulorgeDesmet2N84F": 8}
# domain and velocity of the testcases run through kernel lists
DOMAIN = {"gaussian_rotation_3D": (-1.0, 1.0), "rotation_3D": (-1.0, 1.0), "confined_domain": (0.0, 1.0),
          "hall_periodic": (0.0, 4 * math.pi / 3), "uniform_flow": (0.0, TWO_PI)}


def _case(name, kind, real, n, **more):
    d = {"kind": kind, "real": real, "nx": n[0], "ny": n[1], "nz": n[2]}
    if name:
        d["name"] = name
    d.update(more)
    return d


def listed():
    return [
        # the plain method: rotation on a small bounded grid with inflow SATs, a few steps of a time loop that is
        # run for thousands (latency and the number of launches count)
        _case("rotation_40", "lists", "f64", (40, 40, 40), opset="4thOrder", testcase="gaussian_rotation_3D",
              integrator="SSPRK33", steps=4, hall=False, periodic=False, variable_u=False, dissipation="",
              forms="PRODUCT,CENTRAL,CENTRAL"),
        # one point of the convergence sweeps: periodic Hall problem with a time-dependent velocity
        _case("sweep_60", "lists", "f64", (60, 60, 60), opset="4thOrder", testcase="hall_periodic",
              integrator="CarpenterKennedy2N54", steps=2, hall=True, periodic=True, variable_u=True, dissipation="",
              forms="PRODUCT,CENTRAL,SPLIT"),
        # the Hall problem on a bounded grid (outflow SATs), 6th order, odd size, as in the outflow experiments
        _case("outflow_81", "lists", "f64", (81, 81, 81), opset="6thOrder", testcase="hall_periodic",
              integrator="CarpenterKennedy2N54", steps=1, hall=True, periodic=False, variable_u=True, dissipation="",
              forms="PRODUCT,CENTRAL,CENTRAL"),
        # the headline: periodic Hall time loop with dissipation, cache-sized, both precisions
        _case("hall_128_f64", "uniform", "f64", (128, 128, 128), opset="6thOrder", integrator="CarpenterKennedy2N54",
              steps=4, hall=True, dissipation="HIGH_ORDER", ux=0.0, uy=0.0, uz=0.0, rho=1.0, stated=True),
        _case("hall_128_f32", "uniform", "f32", (128, 128, 128), opset="6thOrder", integrator="CarpenterKennedy2N54",
              steps=4, hall=True, dissipation="HIGH_ORDER", ux=0.0, uy=0.0, uz=0.0, rho=1.0, stated=True),
        # the same beyond the last-level cache
        _case("hall_256_f64", "uniform", "f64", (256, 256, 256), opset="6thOrder", integrator="CarpenterKennedy2N54",
              steps=2, hall=True, dissipation="HIGH_ORDER", ux=0.0, uy=0.0, uz=0.0, rho=1.0, stated=True),
        # a ragged box with a mean flow, three-register scheme, coefficients found uniform by the library
        _case("flow_ragged_f64", "uniform", "f64", (100, 75, 90), opset="4thOrder", integrator="SSPRK33", steps=4,
              hall=True, dissipation="HIGH_ORDER", ux=0.2, uy=-0.1, uz=0.15, rho=1.25, stated=False),
        # a batch of independent solves of uneven sizes
        _case("ensemble_16", "ensemble", "f32", (96, 96, 96), opset="6thOrder", integrator="SSPRK33", steps=10, members=16,
              sizes="32,48,64,96"),
        # gradient of a final-time misfit with respect to the initial field, the velocity and the Hall coefficient
        _case("adjoint_96_f32", "adjoint", "f32", (96, 96, 96), opset="6thOrder", steps=24, snapshots=5),
        # divergence cleaning of a large field with the iteration cap the drivers use
        _case("clean_192_f32", "clean", "f32", (192, 192, 192), opset="4thOrder", laplace="WIDE_STENCIL_DIRICHLET",
              iterations=50),
        # a driver run that records integrals over time and cleans after every step
        _case("series_40", "series", "f64", (40, 40, 40), opset="4thOrder", integrator="CarpenterKennedy2N54", steps=2,
              laplace="WIDE_STENCIL_DIRICHLET", iterations=50),
        # monitoring of a production field
        _case("diagnose_128_f32", "diagnose", "f32", (128, 128, 128), opset="4thOrder", testcase="gaussian_rotation_3D",
              periodic=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, lo, hi, most):
    """Three sizes, each within a factor of about 1.5 of a common one, odd ones among them; at most `most` cells."""
    while True:
        c = _log_int(rng, lo, hi)
        n = tuple(max(lo, min(hi, int(round(c * rng.uniform(0.75, 1.35))))) if rng.random() < 0.6 else c for _ in range(3))
        if n[0] * n[1] * n[2] <= most:
            return n


def draw(rng):
    kind = rng.choice(["uniform", "uniform", "uniform", "lists", "lists", "lists", "ensemble", "adjoint", "clean", "series",
                       "diagnose"])
    real = rng.choice(["f64", "f64", "f32"])
    opset = rng.choice(["2ndOrder", "4thOrder", "6thOrder"])
    form = ",".join([rng.choice(["CENTRAL", "SPLIT", "PRODUCT"]), rng.choice(["ZERO", "CENTRAL", "SPLIT"]),
                     rng.choice(["CENTRAL", "SPLIT", "PRODUCT"])])
    if kind == "uniform":
        n = _grid(rng, 24, 240, 8_000_000)
        hall = rng.random() < 0.8
        flow = not hall or rng.random() < 0.4
        u = [round(rng.uniform(-0.3, 0.3), 3) if flow else 0.0 for _ in range(3)]
        return _case("", kind, real, n, opset=opset, integrator=rng.choice(["SSPRK33", "CarpenterKennedy2N54",
                     "CarpenterKennedy2N54", "ToulorgeDesmet2N84F"]), steps=rng.choice([1, 2, 3]),
                     hall=hall, dissipation=rng.choice(["HIGH_ORDER", "HIGH_ORDER", ""]), ux=u[0], uy=u[1],
                     uz=u[2], rho=round(rng.uniform(0.7, 1.5), 3), stated=rng.random() < 0.7)
    if kind == "lists":
        hall = rng.random() < 0.5
        periodic = rng.random() < (0.6 if hall else 0.25)
        diss = rng.choice(["", "", "HIGH_ORDER", "FIRST_ORDER"])
        opset = rng.choice([opset, opset, opset + "Extended"])
        n = _grid(rng, 24, 120, 700_000)
        return _case("", kind, real, n, opset=opset, testcase="hall_periodic" if hall else
                     rng.choice(["gaussian_rotation_3D", "confined_domain"]),
                     integrator=rng.choice(["SSPRK33", "CarpenterKennedy2N54"]), steps=1, hall=hall, periodic=periodic,
                     variable_u=hall and rng.random() < 0.7, dissipation=diss, forms=form)
    if kind == "ensemble":
        return _case("", kind, real, (0, 0, 0), opset=opset, integrator=rng.choice(["SSPRK33", "CarpenterKennedy2N54"]),
                     steps=4, members=rng.randint(3, 16), sizes=",".join(str(_log_int(rng, 20, 90)) for _ in range(4)))
    if kind == "adjoint":
        return _case("", kind, real, _grid(rng, 24, 96, 700_000), opset=opset, steps=rng.randint(4, 16),
                     snapshots=rng.randint(2, 6))
    if kind == "clean":
        lap = rng.choice(["WIDE_STENCIL_DIRICHLET", "WIDE_STENCIL_DIRICHLET", "NARROW_STENCIL_DIRICHLET"])
        return _case("", kind, real, _grid(rng, 24, 180, 4_000_000), opset=rng.choice(["2ndOrder", "4thOrder"]), laplace=lap,
                     iterations=rng.randint(20, 50))
    if kind == "series":
        return _case("", kind, "f64", _grid(rng, 24, 64, 200_000), opset=rng.choice(["2ndOrder", "4thOrder"]),
                     integrator=rng.choice(["SSPRK33", "CarpenterKennedy2N54"]), steps=rng.randint(1, 3),
                     laplace="WIDE_STENCIL_DIRICHLET", iterations=rng.randint(10, 40))
    return _case("", kind, real, _grid(rng, 24, 200, 6_000_000), opset=rng.choice(["2ndOrder", "4thOrder"]),
                 testcase="gaussian_rotation_3D", periodic=False)


# --- inputs ------------------------------------------------------------------------------------------------------


def _config(case, n=None, dt=1e-3):
    from inductioneq_amd.settings import ProgramConfig

    kind = case["kind"]
    n = n or (case["nx"], case["ny"], case["nz"])
    periodic = kind in ("uniform", "ensemble", "adjoint") or bool(case.get("periodic"))
    tc = {"clean": "gaussian_rotation_3D", "series": "confined_domain"}.get(kind, case.get("testcase", "uniform_flow"))
    lo, hi = DOMAIN[tc]
    if tc != "hall_periodic" and kind == "lists" and periodic:
        hi = lo + 2 * (hi - lo)
    f = case.get("forms", "PRODUCT,CENTRAL,CENTRAL").split(",")
    diss = "HIGH_ORDER" if kind in ("ensemble", "adjoint") else case.get("dissipation") or None
    return ProgramConfig(real=REAL[case["real"]], opset=case["opset"], nx=n[0], ny=n[1], nz=n[2], xmin=lo, xmax=hi, ymin=lo,
                         ymax=hi, zmin=lo, zmax=hi, dt=dt, periodic=periodic,
                         hall=bool(case.get("hall", kind in ("ensemble", "adjoint"))), dissipation=diss, form_uibj=f[0],
                         form_source=f[1], form_ujbi=f[2], testcase=tc, laplace=case.get("laplace"), w_size=256,
                         ux=case.get("ux", 0.0), uy=case.get("uy", 0.0), uz=case.get("uz", 0.0))


def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _axes(cfg):
    a = [lo + torch.arange(m, dtype=torch.float64, device=_dev()) * h for lo, m, h in
         ((cfg.xmin, cfg.nx, cfg.dx), (cfg.ymin, cfg.ny, cfg.dy), (cfg.zmin, cfg.nz, cfg.dz))]
    return a[0][None, None, :], a[1][None, :, None], a[2][:, None, None]


def _waves(cfg, seed, kmax=4, amp=0.1, count=16):
    """Divergence-free random modes |k| <= kmax over the domain's length, amplitudes N(0, amp^2) / |k|^2."""
    rng = np.random.default_rng(seed)
    x, y, z = _axes(cfg)
    L = [cfg.xmax - cfg.xmin, cfg.ymax - cfg.ymin, cfg.zmax - cfg.zmin]
    B = torch.zeros((3, cfg.nz, cfg.ny, cfg.nx), dtype=torch.float64, device=_dev())
    done = 0
    while done < count:
        k = rng.integers(-kmax, kmax + 1, 3)
        k2 = float((k * k).sum())
        if k2 == 0 or k2 > kmax * kmax:
            continue
        kv = k * TWO_PI / np.array(L)
        ab = rng.normal(0.0, amp, (2, 3))
        ab = (ab - (ab @ kv)[:, None] / (kv @ kv) * kv) / k2
        ph = kv[0] * x + kv[1] * y + kv[2] * z
        c, s = torch.cos(ph), torch.sin(ph)
        for i in range(3):
            B[i] += float(ab[0, i]) * c + float(ab[1, i]) * s
        done += 1
    return B


def _hall_dt(h, order, c_hall, bmax, cfl):
    s = {2: 1.0, 4: 1.3722, 6: 1.5860}[order]
    return cfl / (c_hall * bmax * sum((s / d) ** 2 for d in h))


def _gauss(cfg, t=0.0):
    x, y, z = _axes(cfg)
    s, c = math.sin(t), math.cos(t)
    xx, yy = c * x + s * y, -s * x + c * y
    f = torch.exp(-20 * ((xx - 0.5) ** 2 + yy ** 2 + z ** 2))
    bx, by = -40 * yy * f, (40 * xx - 20) * f
    return torch.stack([c * bx - s * by, s * bx + c * by, torch.zeros_like(f)])


def _confined(cfg):
    x, y, z = _axes(cfg)
    sn, cs = (lambda v: torch.sin(math.pi * v)), (lambda v: torch.cos(math.pi * v))
    return torch.stack([sn(x) * cs(y) * cs(z), cs(x) * sn(y) * cs(z), -2 * cs(x) * cs(y) * sn(z)])


def _hall_periodic(cfg, t=0.0, field=True):
    """The travelling wave of the Hall testcase: its field, or its velocity."""
    x, y, z = (a + torch.zeros((cfg.nz, cfg.ny, cfg.nx), dtype=torch.float64, device=_dev()) for a in _axes(cfg))
    n1, al = 1 / math.sqrt(3.0), 0.5
    k = (1 - al * al) / al
    p = al * k * t * n1
    u = torch.stack([torch.cos(k * y + p) + torch.sin(k * z + p), torch.cos(k * z + p) + torch.sin(k * x + p),
                     torch.cos(k * x + p) + torch.sin(k * y + p)])
    return al * u + n1 if field else u


def _velocity(cfg, t=0.0):
    x, y, z = _axes(cfg)
    if cfg.testcase == "gaussian_rotation_3D":
        o = torch.zeros((cfg.nz, cfg.ny, cfg.nx), dtype=torch.float64, device=_dev())
        return torch.stack([o - y, o + x, o])
    if cfg.testcase == "confined_domain":
        return _confined(cfg)
    return _hall_periodic(cfg, t, field=False)


def _start(case, cfg, seed):
    """The initial field of a solve: (3, nz, ny, nx) in 64 bits."""
    kind = case["kind"]
    if kind in ("uniform", "ensemble", "adjoint"):
        B = _waves(cfg, seed)
        B[2] += 1.0
        return B
    base = {"gaussian_rotation_3D": _gauss, "confined_domain": _confined, "hall_periodic": _hall_periodic}[cfg.testcase](cfg)
    if kind == "clean":  # a solenoidal field and the gradient of a random potential
        rng = np.random.default_rng(seed)
        x, y, z = _axes(cfg)
        for _ in range(12):
            k = rng.integers(0, 5, 3)
            c = rng.normal() / max(1.0, float((k * k).sum()))
            w = k * math.pi / 2
            s = -c * torch.sin(w[0] * (x + 1) + w[1] * (y + 1) + w[2] * (z + 1))
            for i in range(3):
                base[i] += s * float(w[i])
        return base
    return base + _waves(cfg, seed, kmax=3, amp=0.02, count=8)


def _setup(case):
    """The configuration of a case with its time step."""
    kind = case["kind"]
    cfg = _config(case)
    h = (cfg.dx, cfg.dy, cfg.dz)
    if kind in ("uniform", "adjoint"):
        cfg.dt = _hall_dt(h, ORDER[case["opset"]], 1.0 / case.get("rho", 1.0), 2.0, 0.4)
        if not cfg.hall:
            cfg.dt = 0.3 * min(h)
    elif kind == "lists":
        cfg.dt = _hall_dt(h, ORDER[case["opset"]], 1.0, 2.5, 0.3) if cfg.hall else 0.3 * min(h)
    elif kind == "series":
        cfg.dt = 0.3 * min(h)
    return cfg


def _members(case):
    """(size, Hall coefficient) of every member."""
    sizes = [int(v) for v in case["sizes"].split(",")]
    return [(sizes[i % len(sizes)], 0.1 + 1.9 * ((7 * i + 3) % 16) / 15.0) for i in range(case["members"])]


def _load(prog, cfg, B):
    f = prog.vector()
    f[:, : cfg.num_nodes] = B.reshape(3, -1).to(prog.torch_dtype)
    return f


def prepare(case, seed):
    from inductioneq_amd.program import Program
    from inductioneq_amd.schedules import rk_schedule

    kind = case["kind"]
    st = {"case": case, "kind": kind}
    if kind == "ensemble":
        from inductioneq_amd.ensemble import Ensemble, MemberSpec

        specs = []
        for n, c in _members(case):
            h = TWO_PI / n
            specs.append(MemberSpec(n, n, n, h, h, h, _hall_dt((h, h, h), ORDER[case["opset"]], c, 2.0, 0.4), rho=1.0 / c))
        prog = Program(_config(case, (32, 32, 32)))
        ens = Ensemble(prog, specs, case["integrator"])
        ens.step(2)  # the launch shape is tuned on the first step
        for i, m in enumerate(specs):
            cfg = _config(case, (m.nx, m.ny, m.nz))
            for r in ens.fields[i]:
                r.zero_()
            ens.fields[i][0][:, : m.nx ** 3] = _start(case, cfg, seed + 1000 * i).reshape(3, -1).to(prog.torch_dtype)
        torch.cuda.synchronize()
        st.update(ens=ens, prog=prog)
        return st
    cfg = _setup(case)
    if kind == "series":
        from inductioneq_amd.harness import HipExecutor

        ex = HipExecutor(cfg)
        ex.prog.use_current_stream()
        b0 = _start(case, cfg, seed).reshape(3, -1).T.contiguous().cpu().numpy()
        u0 = _velocity(cfg).reshape(3, -1).T.contiguous().cpu().numpy()
        st.update(ex=ex, cfg=cfg, b0=b0, u0=u0, rho0=np.ones(cfg.num_nodes))
        return st
    prog = Program(cfg)
    prog.use_current_stream()
    st.update(prog=prog, cfg=cfg, b0=_load(prog, cfg, _start(case, cfg, seed)))
    if kind == "uniform":
        names, nf = rk_schedule(case["integrator"], cfg.hall, False)
        u = _load(prog, cfg, torch.tensor([cfg.ux, cfg.uy, cfg.uz], dtype=torch.float64, device="cuda")[:, None]
                  .expand(3, cfg.num_nodes))
        st["args"] = [st.pop("b0")] + [prog.vector() for _ in range(nf)] + [u, prog.scalar(case["rho"]), prog.time_buffer()]
        st["uniform"] = (cfg.ux, cfg.uy, cfg.uz, case["rho"]) if case["stated"] else None
    elif kind == "lists":
        names, nf = rk_schedule(case["integrator"], cfg.hall, case["variable_u"])
        st["names"] = names * case["steps"]
        st["args"] = [prog.vector() for _ in range(nf + 1)] + [_load(prog, cfg, _velocity(cfg)), prog.scalar(1.0),
                                                               prog.time_buffer()]
    elif kind == "adjoint":
        from inductioneq_amd.adjoint import AdjointSolver

        st["solver"] = AdjointSolver(prog, case["steps"], case["snapshots"])
        st["b0"].requires_grad_(True)
        # the parameters of the model being fitted: velocity and Hall coefficient
        st["p"] = torch.tensor([0.2, -0.1, 0.15, 1.0], dtype=prog.torch_dtype, requires_grad=True)
        st["target"] = _load(prog, cfg, _start(case, cfg, seed + 1))
    elif kind == "clean":
        st["b"], st["phi"] = prog.vector(), prog.scalar()
    return st


# --- one pass ----------------------------------------------------------------------------------------------------


def run(st):
    kind, case = st["kind"], st["case"]
    if kind == "uniform":
        a = st["args"]
        st["prog"].step(case["integrator"], case["steps"], a, uniform=st["uniform"])
        return a[0], a[-1]
    if kind == "lists":  # a solve from the initial data
        a = st["args"]
        a[0].copy_(st["b0"])
        a[-1].zero_()
        st["prog"].run(st["names"], a)
        return a[0], a[-1]
    if kind == "ensemble":
        st["ens"].step(case["steps"])
        return [f[0] for f in st["ens"].fields]
    if kind == "adjoint":
        from inductioneq_amd.adjoint import hall_solve

        cfg = st["cfg"]
        bT = hall_solve(st["b0"], st["p"][:3], st["p"][3], st["solver"])
        loss = (0.5 * cfg.dx * cfg.dy * cfg.dz) * ((bT - st["target"]) ** 2).sum()
        g = torch.autograd.grad(loss, [st["b0"], st["p"]])
        return {"b": bT.detach(), "gb": g[0], "gp": g[1]}
    if kind == "clean":
        st["b"].copy_(st["b0"])
        r = st["prog"].clean_div_cg(st["b"], phi=st["phi"], abs_threshold=1e-3, max_iterations=case["iterations"])
        return {"b": st["b"], "phi": st["phi"], "iterations": r["iterations"]}
    if kind == "series":
        from inductioneq_amd.harness import compute_numerical_solution

        cfg = st["cfg"]
        r = compute_numerical_solution(cfg, st["ex"], case["integrator"], st["b0"], st["u0"], st["rho0"], case["steps"],
                                       case["steps"] * cfg.dt, save_integrals_over_time=True,
                                       divergence_cleaning=(1e-3, case["iterations"]))
        return {"b": r["field_b"], "energy": r["energy_over_time"], "div": r["L2error_divB_over_time"],
                "error": r["L2error_B_over_time"], "iterations": [int(i) for i in r["cg_iterations"]]}
    d = st["prog"].diagnostics(st["b0"], 0.1)
    return [d["energy"], d["divergence_norm"], d["error_norm"]]


# --- what a pass cannot do without -------------------------------------------------------------------------------


def _stage_work(case, cells, stages):
    """Values moved and operations of RK stages: the state (and velocity field) read, the registers read and written."""
    r = ORDER[case["opset"]] // 2
    two_n = "2N" in case["integrator"]
    first = 4 * 3 if two_n else 8  # vector fields per stage: B, b2 in and out; three registers: 8/3 on average
    words = cells * stages * (first if two_n else 8)
    ops = 0
    if case.get("hall", True):
        ops += 12 * 4 * r + 9 + 9  # curl B, J x B, curl E
    if case.get("dissipation", "HIGH_ORDER"):
        ops += 9 * 3 * r
    if case["kind"] == "lists":
        words += cells * stages * (0 if case["variable_u"] else 3)  # a static velocity field is read
        ops += 9 * 3 * 4 * r
    elif case.get("ux") or case.get("uy") or case.get("uz"):
        ops += 9 * 4 * r
    return words, cells * stages * (ops + 12)


def work(case):
    kind = case["kind"]
    rb = 8 if case["real"] == "f64" else 4
    cells = case["nx"] * case["ny"] * case["nz"]
    r = ORDER[case["opset"]] // 2
    if kind in ("uniform", "lists"):
        w, f = _stage_work(case, cells, case["steps"] * STAGES[case["integrator"]])
    elif kind == "ensemble":
        w, f = _stage_work(case, sum(n ** 3 for n, _ in _members(case)), case["steps"] * STAGES[case["integrator"]])
    elif kind == "adjoint":  # forward, the two stage inputs of every reversed step, three transposed stages
        k = dict(case, integrator="SSPRK33", ux=0.2)
        w, f = _stage_work(k, cells, 8 * case["steps"])
    elif kind == "clean":  # per iteration: u, r in, u', q out; phi, u', r, q in, phi, r out
        w, f = cells * (10 * case["iterations"] + 8), cells * case["iterations"] * (3 * 2 * (4 * r + 1) + 12)
    elif kind == "series":
        w, f = _stage_work(dict(case, kind="lists", variable_u=False, hall=False, dissipation=""), cells,
                           case["steps"] * STAGES[case["integrator"]])
        w += cells * case["steps"] * (10 * case["iterations"] + 8 + 8)
        f += cells * case["steps"] * case["iterations"] * (3 * 2 * (4 * r + 1) + 12)
    else:
        w, f = 3 * cells, cells * (3 * 4 * r + 60)
    return {"bytes": float(w * rb), "flops": float(f)}


# --- the same in 64 bits, without the library ----------------------------------------------------------------------

# Central rows at offsets 1..r; the classical boundary closures of orders 2 and 4 (rows from the left face) and
# the inverse norm weights (Mattsson and Nordstrom, J. Comput. Phys. 199, 2004)
_CENTRAL = {2: [1 / 2], 4: [2 / 3, -1 / 12], 6: [3 / 4, -3 / 20, 1 / 60]}
_CLOSURE = {2: [[-1, 1]],
            4: [[-24 / 17, 59 / 34, -4 / 17, -3 / 34], [-1 / 2, 0, 1 / 2], [4 / 43, -59 / 86, 0, 59 / 86, -4 / 43],
                [3 / 98, 0, -59 / 98, 0, 32 / 49, -4 / 49]]}
_MINV = {2: [2.0], 4: [48 / 17, 48 / 59, 48 / 43, 48 / 49]}


def _dmat(order, n, h, periodic):
    D = torch.zeros((n, n), dtype=torch.float64)
    c = _CENTRAL[order]
    for i in range(n):
        for k, v in enumerate(c, 1):
            for j, w in ((i + k, v), (i - k, -v)):
                if periodic:
                    D[i, j % n] += w
                elif 0 <= j < n:
                    D[i, j] = w
    if not periodic:
        for i, row in enumerate(_CLOSURE[order]):
            D[i], D[n - 1 - i] = 0, 0
            for j, v in enumerate(row):
                D[i, j], D[n - 1 - i, n - 1 - j] = v, -v
    return (D / h).to(_dev())


def _smat(order, n):
    """Periodic high-order dissipation of one direction: (-1)^(r+1) times the r-th difference squared."""
    r = order // 2
    w = np.array([1.0])
    for _ in range(order):
        w = np.convolve(w, [1.0, -1.0])
    S = torch.zeros((n, n), dtype=torch.float64)
    sgn = -1.0 if w[r] > 0 else 1.0
    for i in range(n):
        for k in range(-r, r + 1):
            S[i, (i + k) % n] += sgn * w[k + r]
    return S.to(_dev())


def _along(M, f, d):
    """M applied along x (d = 0), y or z of f[..., z, y, x]."""
    if d == 0:
        return f @ M.T
    if d == 1:
        return M @ f
    return (M @ f.reshape(f.shape[:-3] + (f.shape[-3], -1))).reshape(f.shape)


class _Exact:
    def __init__(self, case, cfg):
        o = ORDER[case["opset"]]
        self.cfg, self.per, self.order = cfg, cfg.periodic, o
        self.h = (cfg.dx, cfg.dy, cfg.dz)
        self.n = (cfg.nx, cfg.ny, cfg.nz)
        self.D = [_dmat(o, m, h, cfg.periodic) for m, h in zip(self.n, self.h)]
        self.S = [_smat(o, m) for m in self.n] if cfg.dissipation == "HIGH_ORDER" else None

    def curl(self, f):
        d = lambda k, c: _along(self.D[k], f[c], k)  # noqa: E731
        return torch.stack([d(1, 2) - d(2, 1), d(2, 0) - d(0, 2), d(0, 1) - d(1, 0)])

    def div(self, f):
        return sum(_along(self.D[k], f[k], k) for k in range(3))

    def weights(self):
        w = 1.0
        for k, (m, h) in enumerate(zip(self.n, self.h)):
            v = torch.full((m,), h, dtype=torch.float64, device=_dev())
            if not self.per:
                for i, q in enumerate(_MINV[self.order]):
                    v[i], v[m - 1 - i] = h / q, h / q
            w = w * v.reshape([-1 if k == 2 - j else 1 for j in range(3)])
        return w

    def faces(self, d):
        """Masks of the two faces of direction d."""
        lo = torch.zeros(self.n[d], dtype=torch.float64, device=_dev())
        hi = lo.clone()
        lo[0], hi[-1] = 1, 1
        s = [-1 if d == 2 - j else 1 for j in range(3)]
        return lo.reshape(s), hi.reshape(s)

    def rhs(self, B, u, t, rho, bound=None):
        cfg = self.cfg
        D, r = self.D, 0
        if u is not None:
            for d in range(3):
                A = lambda f: _along(D[d], f, d)  # noqa: E731, B023
                bd, ud = B[d], u[d]
                if cfg.form_uibj == "CENTRAL":
                    f = A(bd * u)
                elif cfg.form_uibj == "SPLIT":
                    f = 0.5 * (bd * A(u) + u * A(bd) + A(bd * u))
                else:
                    f = u * A(bd) + bd * A(u)
                if cfg.form_source == "CENTRAL":
                    f = f - u * A(bd)
                elif cfg.form_source == "SPLIT":
                    f = f - 0.5 * (u * A(bd) + A(bd * u) - bd * A(u))
                if cfg.form_ujbi == "CENTRAL":
                    f = f - A(ud * B)
                elif cfg.form_ujbi == "SPLIT":
                    f = f - 0.5 * (ud * A(B) + B * A(ud) + A(ud * B))
                else:
                    f = f - (ud * A(B) + B * A(ud))
                r = r + f
        if cfg.hall:
            J = self.curl(B) / rho
            for d in range(3):
                r = r + _along(D[d], J[d] * B - B[d] * J, d)
        if not self.per:
            m0 = _MINV[self.order][0]
            for d in range(3):
                lo, hi = self.faces(d)
                if cfg.hall:
                    tv = 0.5 * u[d] - J[d]
                    s1 = hi * (tv < 0) - lo * (tv > 0)
                    r = r + (m0 / self.h[d]) * (s1 * tv * B + (hi - lo) * B[d] * J)
                else:
                    s = hi * (u[d] < 0) - lo * (u[d] > 0)
                    r = r + (m0 / self.h[d]) * s * u[d] * (B - bound(t))
        if self.S is not None:
            r = r + cfg.ho_factor * sum(_along(self.S[d], B, d) for d in range(3))
        return r

    def step(self, integrator, B, t, dt, u, rho=1.0, bound=None):
        """One RK step; u(t) is the velocity (or None)."""
        F = lambda b, s: self.rhs(b, u(s), s, rho, bound)  # noqa: E731
        if integrator == "SSPRK33":
            b2 = B + dt * F(B, t)
            b3 = 0.75 * B + 0.25 * b2 + 0.25 * dt * F(b2, t + dt)
            return B / 3 + 2 / 3 * b3 + 2 / 3 * dt * F(b3, t + 0.5 * dt)
        if integrator == "CarpenterKennedy2N54":
            A = [0.0, -567301805773 / 1357537059087, -2404267990393 / 2016746695238, -3550918686646 / 2091501179385,
                 -1275806237668 / 842570457699]
            Bc = [1432997174477 / 9575080441755, 5161836677717 / 13612068292357, 1720146321549 / 2090206949498,
                  3134564353537 / 4481467310338, 2277821191437 / 14882151754819]
            c = [0.0, 1432997174477 / 9575080441755, 2526269341429 / 6820363962896, 2006345519317 / 3224310063776,
                 2802321613138 / 2924317926251]
        else:  # ToulorgeDesmet2N84F, for velocities that do not depend on time
            A = [0.0, -0.5534431294501569, 0.01065987570203490, -0.5515812888932000, -1.885790377558741, -5.701295742793264,
                 2.113903965664793, -0.5339578826675280]
            Bc = [0.08037936882736950, 0.5388497458569843, 0.01974974409031960, 0.09911841297339970, 0.7466920411064123,
                  1.679584245618894, 0.2433728067008188, 0.1422730459001373]
            c = [0.0] * 8
        k = torch.zeros_like(B)
        for a, b, s in zip(A, Bc, c):
            k = a * k + dt * F(B, t + s * dt)
            B = B + b * k
        return B

    def clean(self, B, iterations, threshold, narrow=False):
        """CG on -Lap phi = div B with 0 on the faces, then B + grad phi."""
        inner = torch.ones((self.n[2], self.n[1], self.n[0]), dtype=torch.float64, device=_dev())
        for d in range(3):
            lo, hi = self.faces(d)
            inner = inner * (1 - lo) * (1 - hi)
        if narrow:
            M = []
            for m, h in zip(self.n, self.h):
                L = 2 * torch.eye(m, dtype=torch.float64)
                L -= torch.diag(torch.ones(m - 1, dtype=torch.float64), 1) + torch.diag(torch.ones(m - 1, dtype=torch.float64), -1)
                M.append((L / h ** 2).to(_dev()))
        else:
            M = [-(D @ D) for D in self.D]
        lap = lambda f: inner * sum(_along(M[d], f, d) for d in range(3))  # noqa: E731
        r = inner * self.div(B)
        phi, u, old, it = torch.zeros_like(r), torch.zeros_like(r), 1.0, 0
        rr = float((r * r).sum())
        while rr > threshold ** 2 and it < iterations:
            u = (rr / old) * u + r
            q = lap(u)
            a = rr / float((u * q).sum())
            phi, r, old = phi + a * u, r - a * q, rr
            rr = float((r * r).sum())
            it += 1
        return B + torch.stack([_along(self.D[k], phi, k) for k in range(3)]), phi


def _rounded(case, v):
    return v.to(torch.float32).double() if case["real"] == "f32" else v


def _padded(cfg, v):
    """(c, nz, ny, nx) -> the library's layout with zero padding."""
    pad = (cfg.num_nodes_pad + 63) // 64 * 64
    out = torch.zeros((v.shape[0], pad), dtype=torch.float64, device=v.device)
    out[:, : cfg.num_nodes] = v.reshape(v.shape[0], -1)
    return out


def exact(case, seed):
    kind = case["kind"]
    bounded = kind in ("clean", "series", "diagnose") or (kind == "lists" and not case["periodic"])
    if "Extended" in case["opset"] and (bounded or kind == "lists"):
        return None
    if kind == "lists" and (case["dissipation"] == "FIRST_ORDER" or (bounded and case["dissipation"])):
        return None
    if bounded and ORDER[case["opset"]] == 6:
        return None
    if kind == "clean" and case["laplace"].startswith("NARROW") and ORDER[case["opset"]] != 2:
        return None
    if kind == "ensemble":
        out = []
        for i, (n, c) in enumerate(_members(case)):
            cfg = _config(case, (n, n, n))
            h = TWO_PI / n
            dt = _hall_dt((h, h, h), ORDER[case["opset"]], c, 2.0, 0.4)
            B, X = _rounded(case, _start(case, cfg, seed + 1000 * i)), _Exact(case, cfg)
            for _ in range(case["steps"]):
                B = X.step(case["integrator"], B, 0.0, dt, lambda t: None, 1.0 / c)
            out.append(_member_layout(B))
        return out
    cfg = _setup(case)
    X = _Exact(case, cfg)
    B = _rounded(case, _start(case, cfg, seed))
    if kind in ("uniform", "lists"):
        if kind == "uniform":
            if cfg.ux or cfg.uy or cfg.uz:
                v = torch.tensor([cfg.ux, cfg.uy, cfg.uz], dtype=torch.float64, device=_dev())[:, None, None, None]
                v = v.expand(B.shape)
                u = lambda t: v  # noqa: E731
            else:
                u = lambda t: None  # noqa: E731
            rho, bound = case["rho"], None
        else:
            v = _rounded(case, _velocity(cfg))
            u = (lambda t: _velocity(cfg, t)) if case["variable_u"] else (lambda t: v)
            rho, bound = 1.0, (lambda t: _gauss(cfg, t) if cfg.testcase == "gaussian_rotation_3D" else _confined(cfg))
        for k in range(case["steps"]):
            B = X.step(case["integrator"], B, k * cfg.dt, cfg.dt, u, rho, bound)
        t = case["steps"] * cfg.dt
        return _padded(cfg, B), torch.tensor([t, t], dtype=torch.float64)
    if kind == "adjoint":
        target = _rounded(case, _start(case, cfg, seed + 1))
        B.requires_grad_(True)
        par = torch.tensor([0.2, -0.1, 0.15, 1.0], dtype=torch.float64).requires_grad_(True)
        pv = _rounded(case, par).to(_dev())
        uu, c = pv[:3, None, None, None].expand(B.shape), pv[3]
        b = B
        for _ in range(case["steps"]):
            b = X.step("SSPRK33", b, 0.0, cfg.dt, lambda t: uu, 1.0 / c)
        loss = (0.5 * cfg.dx * cfg.dy * cfg.dz) * ((b - target) ** 2).sum()
        g = torch.autograd.grad(loss, [B, par])
        return {"b": _padded(cfg, b.detach()), "gb": _padded(cfg, g[0]), "gp": g[1]}
    if kind == "clean":
        b, phi = X.clean(B, case["iterations"], 1e-3, case["laplace"].startswith("NARROW"))
        return {"b": _padded(cfg, b), "phi": _padded(cfg, phi[None])[0], "iterations": None}
    if kind == "series":
        w, ana = X.weights(), _confined(cfg)
        E, V, R = [], [], []

        def integrals():
            E.append(float((w * (B * B).sum(0)).sum()))
            V.append(math.sqrt(float((w * X.div(B) ** 2).sum())))
            R.append(math.sqrt(float((w * ((B - ana) ** 2).sum(0)).sum())))

        v = _velocity(cfg)
        for k in range(case["steps"]):
            integrals()
            B = X.step(case["integrator"], B, k * cfg.dt, cfg.dt, lambda t: v, 1.0, lambda t: ana)
            B, _ = X.clean(B, case["iterations"], 1e-3)
        integrals()
        return {"b": B.reshape(3, -1).T.contiguous(), "energy": np.array(E), "div": np.array(V), "error": np.array(R),
                "iterations": None}
    w = X.weights()
    d = X.div(B)
    e = B - _gauss(cfg, 0.1)
    return [float((w * (B * B).sum(0)).sum()), math.sqrt(float((w * d * d).sum())), math.sqrt(float((w * (e * e).sum(0)).sum()))]


def _member_layout(B):
    n = B[0].numel()
    out = torch.zeros((3, (n + 63) // 64 * 64), dtype=torch.float64, device=B.device)
    out[:, :n] = B.reshape(3, -1)
    return out
