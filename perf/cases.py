"""The work that programs have this library do, as timed cases.

Every case runs through the Python binding (laboetie_amd.lbx), which is the
C-ABI of include/lbx.h one to one.  Five kinds of use ("path"):

  solve    one lattice from rest: equilibration, then moment propagation of
           one tracer, with the flow, VACF, D_eff and P read back (the whole
           job of one lb.in on a context that the program keeps);
  flow     the equilibration alone, the density and flux read back
           (permeability runs);
  tracers  moment propagation of 1 to 4 tracers on a flow that the program
           already has, VACF and D_eff read back;
  program  what the Fortran driver does with one lb.in, host arrays in and
           out: create, upload the state, equilibrate, download it, moment
           propagation from that flow in chunks that overlap with the host;
  batch    many lattices admitted to one batch engine and advanced together
           until all are done (2-D chromatography cells of two sizes, or
           served 3-D requests of mixed sizes and geometries).

A pass takes fewer time steps than a production run of the same lattice (a
thousand instead of several thousand), so that the smallest and the largest
lattices can be timed in one sitting.
"""
import math

import numpy as np
import torch

from laboetie_amd import lbx

PREC = {"fp64": lbx.PREC_FP64, "fp32_shift": lbx.PREC_FP32_SHIFT, "fp32_store": lbx.PREC_FP32_STORE}
DB = 0.01           # tracer diffusion coefficient of every configuration
TARGET = 0.0        # equilibrations of a fixed number of steps, as the precision runs take them
FLOW_STEPS = 200    # LB steps behind the flow that a "tracers" case starts from
CHUNK = 256         # MP steps per begun chunk of the driver's propagate()


def _case(name, path, geom, lx, ly, lz, prec="fp64", tau=1.0, force=1e-6, lb=0, mp=0, tracers=1, porosity=0.6,
          sigma=4.0, count=1):
    c = dict(path=path, geom=geom, lx=lx, ly=ly, lz=lz, prec=prec, tau=tau, force=force, lb_steps=lb, mp_steps=mp,
             tracers=tracers, porosity=porosity, sigma=sigma, count=count)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # the smallest lattice anybody runs: the validation slit against Poiseuille (544 nodes)
        _case("slit_4x4x34", "solve", "slit", 4, 4, 34, force=1e-5, lb=2000, mp=1000),
        # one 2-D chromatography cell solved by itself
        _case("disks_1x50x50", "solve", "disks", 1, 50, 50, force=1e-5, lb=1000, mp=1000, count=4),
        # a small served request solved by itself, odd size, in the accurate FP32-storage form
        _case("cylinder_45_fp32_store", "solve", "cylinder", 45, 45, 45, prec="fp32_store", lb=500, mp=500),
        # the Fortran program's run of a BCC cell, host arrays in and out
        _case("program_bcc_64", "program", "bcc", 64, 64, 64, lb=400, mp=512),
        # the headline lattice: its flow, and its three adsorbing tracers
        _case("flow_bcc_128", "flow", "bcc", 128, 128, 128, lb=1000),
        _case("tracers3_bcc_128", "tracers", "bcc", 128, 128, 128, mp=1000, tracers=3),
        # a ragged porous sample with one tracer, as the driver propagates it
        _case("tracer1_random_150x97x121", "tracers", "random", 150, 97, 121, tau=0.8, mp=500),
        # the large porous medium (correlation length 8, porosity 0.6) in FP64: flow and tracer
        _case("flow_random_256", "flow", "random", 256, 256, 256, tau=0.8, lb=300, sigma=8.0),
        _case("tracer1_random_256", "tracers", "random", 256, 256, 256, tau=0.8, mp=300, sigma=8.0),
        # the largest served request size in the fast FP32-storage form
        _case("flow_random_192_fp32_shift", "flow", "random", 192, 192, 192, prec="fp32_shift", tau=0.8, lb=600),
        # the chromatography batch: 1x50x50 and 1x100x100 cells in equal parts
        _case("batch_1024_disks", "batch", "disks", 1, 100, 100, force=1e-5, lb=256, mp=256, count=1024),
        # a served mix of 3-D requests, FP32-shift, sizes log-uniform up to lx
        _case("batch_8_mixed_fp32_shift", "batch", "mixed", 96, 96, 96, prec="fp32_shift", lb=256, mp=192, count=8),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    path = rng.choice(["solve", "solve", "program", "flow", "flow", "tracers", "tracers", "batch"])
    prec = rng.choice(["fp64", "fp64", "fp32_shift", "fp32_store"])
    tau = rng.choice([1.0, 1.0, 0.8, rng.uniform(0.6, 1.5)])
    force = _log_uniform(rng, 1e-7, 1e-5)
    porosity, sigma = rng.uniform(0.4, 0.8), rng.choice([4.0, 8.0])
    if path == "batch":
        if rng.random() < 0.5:
            n = int(_log_uniform(rng, 16, 900))
            side = rng.choice([50, 64, 75, 100])
            return _case(None, path, "disks", 1, side, side, prec, tau, 1e-5, rng.randrange(100, 256),
                         rng.randrange(100, 256), 1, porosity, sigma, n)
        side = rng.randrange(48, 90)
        return _case(None, path, "mixed", side, side, side, prec, tau, force, rng.randrange(100, 256),
                     rng.randrange(100, 192), 1, porosity, sigma, rng.randrange(3, 9))
    lo, hi = {"solve": (8, 64), "program": (12, 72), "flow": (40, 220), "tracers": (40, 220)}[path]
    geom = rng.choice(["slit", "cylinder", "bcc", "random", "random"] + (["disks"] if path == "solve" else []))
    n = max(lo, min(hi, int(round(_log_uniform(rng, lo, hi)))))
    if geom == "disks":
        lx, ly, lz = 1, max(24, n), max(24, int(n * rng.uniform(0.6, 1.6)))
    elif geom == "random":  # any box
        lx, ly, lz = (max(8, min(hi, int(n * rng.uniform(0.7, 1.4)))) for _ in range(3))
    elif geom == "slit":
        lx, ly, lz = max(4, int(n * rng.uniform(0.3, 1.0))), max(4, int(n * rng.uniform(0.3, 1.0))), n
    elif geom == "cylinder":
        lx, ly, lz = n, n, max(4, int(n * rng.uniform(0.5, 1.2)))
    else:
        lx = ly = lz = n
    nodes = lx * ly * lz
    lb = max(100, min(900, int(1.5e9 / nodes)))
    mp = max(100, min(900, int(1.0e9 / nodes)))
    return _case(None, path, geom, lx, ly, lz, prec, tau, force, lb if path != "tracers" else 0,
                 mp if path != "flow" else 0, rng.choice([1, 1, 2, 3, 4]) if path == "tracers" else 1, porosity,
                 sigma, rng.randrange(1, 9))


# ------------------------------------------------------------------ inputs
def _dims(c):
    return c["lx"], c["ly"], c["lz"]


def _grid(lx, ly, lz):
    """1-based node coordinates, broadcastable to (lz, ly, lx)."""
    a = [torch.arange(1, n + 1, device="cuda", dtype=torch.float64) for n in (lx, ly, lz)]
    return a[0][None, None, :], a[1][None, :, None], a[2][:, None, None]


def _slit(lx, ly, lz):
    s = torch.zeros((lz, ly, lx), dtype=torch.bool, device="cuda")
    s[0] = s[-1] = True
    return s


def _cylinder(lx, ly, lz):
    x, y, _ = _grid(lx, ly, 1)
    r2 = (x - (lx + 1) / 2.0) ** 2 + (y - (ly + 1) / 2.0) ** 2
    return (r2 >= ((lx - 1) / 2.0) ** 2).expand(lz, ly, lx).contiguous()


def _bcc(lx, ly, lz):
    x, y, z = _grid(lx, ly, lz)
    rad2 = ((lx - 1) * math.sqrt(3.0) / 4.0) ** 2
    s = torch.zeros((lz, ly, lx), dtype=torch.bool, device="cuda")
    mid = (lx + 1) / 2.0
    for cx, cy, cz in [(i, j, k) for i in (1, lx) for j in (1, ly) for k in (1, lz)] + [(mid, mid, mid)]:
        s |= (x - cx) ** 2 + (y - cy) ** 2 + (z - cz) ** 2 <= rad2
    return s


def _random(lx, ly, lz, sigma, porosity, seed):
    """Gaussian-filtered white noise, the lowest porosity fraction fluid."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    f = torch.fft.rfftn(torch.randn((lz, ly, lx), generator=g, device="cuda"))
    for axis, n in enumerate((lz, ly, lx)):
        k = torch.arange(f.shape[axis], device="cuda", dtype=torch.float32)
        k = torch.minimum(k, n - k) / n
        shape = [1, 1, 1]
        shape[axis] = -1
        f = f * torch.exp(-2.0 * (math.pi * sigma * k) ** 2).reshape(shape)
    f = torch.fft.irfftn(f, s=(lz, ly, lx))
    cut = torch.sort(f.reshape(-1)).values[max(0, int(porosity * f.numel()) - 1)]
    return f > cut


def _disks(ly, lz, n, rng):
    """Up to n non-touching disks of radius 5 in a periodic ly x lz cell."""
    s = torch.zeros((lz, ly, 1), dtype=torch.bool, device="cuda")
    _, y, z = _grid(1, ly, lz)
    placed = []
    for _ in range(200):
        if len(placed) == n:
            break
        p = (rng.uniform(1, ly + 1), rng.uniform(1, lz + 1))
        gap = [math.hypot(min(abs(p[0] - q[0]), ly - abs(p[0] - q[0])), min(abs(p[1] - q[1]), lz - abs(p[1] - q[1])))
               for q in placed]
        if all(d > 10.0 for d in gap):
            placed.append(p)
    for py, pz in placed:
        dy, dz = (y - py).abs(), (z - pz).abs()
        s |= torch.minimum(dy, ly - dy) ** 2 + torch.minimum(dz, lz - dz) ** 2 <= 25.0
    return s


def _solid(geom, lx, ly, lz, c, rng):
    if geom == "slit":
        return _slit(lx, ly, lz)
    if geom == "cylinder":
        return _cylinder(lx, ly, lz)
    if geom == "bcc":
        return _bcc(lx, ly, lz)
    if geom == "disks":
        return _disks(ly, lz, int(rng.integers(1, 9)) if c["path"] == "batch" else c["count"], rng)
    return _random(lx, ly, lz, c["sigma"], c["porosity"], int(rng.integers(1, 2 ** 31)))


# the open axis of each geometry
_AXIS = {"slit": 0, "cylinder": 2, "bcc": 2, "random": 0, "disks": 1}


def _force(geom, size, rng):
    f = [0.0, 0.0, 0.0]
    f[_AXIS[geom]] = size * float(rng.uniform(0.8, 1.25))
    return f


def _adsorption(n, rng):
    """(ka, kd) of n tracers: adsorption free energies in [-3, 0] kT."""
    pairs = [lbx.ka_kd_from_dF(float(rng.uniform(-3.0, 0.0))) for _ in range(n)]
    return [p[0] for p in pairs], [p[1] for p in pairs]


def _inputs(c, seed):
    """One lattice's inputs: solid mask (lz, ly, lx), force, ka, kd."""
    rng = np.random.default_rng([seed, 11])
    solid = _solid(c["geom"], *_dims(c), c, rng)
    return solid, _force(c["geom"], c["force"], rng), *_adsorption(c["tracers"], rng)


def _requests(c, seed):
    """The lattices of a batch case: (geom, dims, solid, force, ka, kd) each.
    "disks": cells of the full and of half the side in turn; "mixed": served
    requests, cubic, sides log-uniform from a third of lx up to lx."""
    rng = np.random.default_rng([seed, 13])
    shape_rng = np.random.default_rng(17)  # a mix's sizes belong to the case, not to the seed
    out = []
    for k in range(c["count"]):
        if c["geom"] == "disks":
            geom, dims = "disks", (1, c["ly"] if k % 2 else c["ly"] // 2, c["lz"] if k % 2 else c["lz"] // 2)
        else:
            n = int(round(math.exp(shape_rng.uniform(math.log(c["lx"] / 3), math.log(c["lx"])))))
            geom, dims = ("slit", "cylinder", "bcc", "random")[k % 4], (n, n, n)
        solid = _solid(geom, *dims, c, rng)
        ka, kd = _adsorption(1, rng)
        out.append((geom, dims, solid, _force(geom, c["force"], rng), ka[0], kd[0]))
    return out


def _nature(solid):
    return solid.to(torch.int8).cpu().numpy().reshape(-1)


def prepare(case, seed):
    c = case
    s = {"case": c}
    if c["path"] == "batch":
        reqs = _requests(c, seed)
        s["reqs"] = [(dims, _nature(solid), F, ka, kd) for _, dims, solid, F, ka, kd in reqs]
        nodes = sum(-(-int((nat == 0).sum()) // 256) * 256 for _, nat, _, _, _ in s["reqs"])
        box = sum(nat.size for _, nat, _, _, _ in s["reqs"])
        s["batch"] = lbx.Batch(nodes + 256, box + 256, len(reqs), precision=PREC[c["prec"]])
        return s
    solid, s["F"], s["ka"], s["kd"] = _inputs(c, seed)
    s["nature"] = _nature(solid)
    if c["path"] == "program":
        # the rest state as init_simu leaves it, in the program's own arrays
        _, w, _, _, _ = lbx.d3q19_tables()
        fluid = (s["nature"] == 0).astype(np.float64)
        s["n"], s["rho"] = np.outer(w, fluid).reshape(-1), fluid
        s["j"] = np.zeros((3, fluid.size))
        return s
    s["lattice"] = L = lbx.Lattice(_dims(c), s["nature"], c["tau"], precision=PREC[c["prec"]])
    if c["path"] == "tracers":
        L.init_rest(1.0)
        L.equilibrate(s["F"], TARGET, max_steps=FLOW_STEPS, trace_cap=1)
    return s


# ------------------------------------------------------------------ one pass
def _run_solve(c, s):
    L = s["lattice"]
    L.init_rest(1.0)
    e = L.equilibrate(s["F"], TARGET, max_steps=c["lb_steps"], trace_cap=c["lb_steps"])
    v0 = L.mp_init(s["F"], DB, s["ka"][0], s["kd"][0])
    m = L.mp_run(c["mp_steps"])
    d = L.mp_deff()
    _, rho, j = L.get_state(populations=False)
    P, Pa = L.mp_get()
    return {"l2err": e["l2err"], "rho": rho, "j": j, "vacf0": v0, "vacf": m["vacf"], "deff": d, "P": P, "Pa": Pa}


def _run_flow(c, s):
    L = s["lattice"]
    L.init_rest(1.0)
    e = L.equilibrate(s["F"], TARGET, max_steps=c["lb_steps"], trace_cap=c["lb_steps"])
    _, rho, j = L.get_state(populations=False)
    return {"l2err": e["l2err"], "rho": rho, "j": j}


def _run_tracers(c, s):
    L = s["lattice"]
    v0 = L.mp_init_batch(s["F"], DB, s["ka"], s["kd"])
    m = L.mp_run(c["mp_steps"])
    return {"vacf0": v0, "vacf": m["vacf"], "deff": L.mp_deff()}


def _run_program(c, s):
    with lbx.Lattice(_dims(c), s["nature"], c["tau"], precision=PREC[c["prec"]]) as L:
        L.set_state(s["n"], s["rho"], s["j"])
        L.equilibrate_begin(s["F"], TARGET, max_steps=c["lb_steps"])
        L.equilibrate_advance()
        n, rho, j = L.get_state()
        v0 = L.mp_init(s["F"], DB, s["ka"][0], s["kd"][0], flow=(rho, j))
        vacf, left = [], c["mp_steps"]
        while left > 0:
            L.mp_run_start(min(CHUNK, left), stop_on_convergence=True)
            r = L.mp_run_wait()
            vacf.append(r["vacf"])
            left -= r["steps"]
            if r["converged"]:
                break
        return {"l2err": L.l2err_trace(), "n": n, "rho": rho, "j": j, "vacf0": v0, "vacf": np.concatenate(vacf),
                "deff": L.mp_deff()}


def _run_batch(c, s):
    B = s["batch"]
    ids = [B.add(dims, nat, c["tau"], 1.0, F, TARGET, DB, ka, kd, c["mp_steps"], max_lb_steps=c["lb_steps"])
           for dims, nat, F, ka, kd in s["reqs"]]
    while B.round(128, 128):
        pass
    res = [B.result(i, vacf_rows=c["mp_steps"] + 1) for i in ids]
    for i in ids:
        B.remove(i)
    return {"deff": np.stack([r["deff"] for r in res]), "vacf": np.stack([r["vacf"] for r in res])}


_RUN = {"solve": _run_solve, "flow": _run_flow, "tracers": _run_tracers, "program": _run_program, "batch": _run_batch}


def run(state):
    return _RUN[state["case"]["path"]](state["case"], state)


# ------------------------------------------------------------------ work
def _fluid_nodes(c):
    """Fluid nodes per case: exact for the named geometries, the porosity for
    the random medium, the cell less its disks for the cells."""
    def one(geom, lx, ly, lz):
        n = lx * ly * lz
        if geom == "slit":
            return n * (lz - 2) / lz
        if geom == "cylinder":
            return n * math.pi / 4 * ((lx - 1) / lx) ** 2
        if geom == "bcc":
            return n * (1 - math.pi * math.sqrt(3.0) / 8)
        if geom == "disks":
            return n - math.pi * 25 * min(4.5 if c["path"] == "batch" else c["count"], n / 200)
        return n * c["porosity"]
    if c["path"] != "batch":
        return one(c["geom"], *_dims(c))
    if c["geom"] == "disks":
        half = one("disks", 1, c["ly"] // 2, c["lz"] // 2)
        return (half + one("disks", *_dims(c))) * c["count"] / 2
    rng = np.random.default_rng(17)
    sides = [int(round(math.exp(rng.uniform(math.log(c["lx"] / 3), math.log(c["lx"]))))) for _ in range(c["count"])]
    return sum(one(("slit", "cylinder", "bcc", "random")[k % 4], n, n, n) for k, n in enumerate(sides))


def work(case):
    """Bytes and operations of the time steps, per fluid node and step: an LB
    step reads and writes 19 populations; an MP step reads the density and
    flow its probabilities follow from (4 values) and reads and writes 3
    values of P per tracer.  Operations: about 650 of a collision with its
    moments, and per MP step 18 probabilities (8 each) and 36 multiply-adds'
    worth per tracer and component."""
    c = case
    nf, b = _fluid_nodes(c), 8 if c["prec"] == "fp64" else 4
    T = c["tracers"]
    lb, mp = c["lb_steps"], c["mp_steps"]
    return {"bytes": nf * (lb * 38 * b + mp * (32 + 48 * T)), "flops": nf * (lb * 650 + mp * (144 + 114 * T))}


# ------------------------------------------------------------------ 64 bits
_C = [(0, 0, 0), (1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1), (1, 1, 0), (-1, 1, 0),
      (1, -1, 0), (-1, -1, 0), (1, 0, 1), (-1, 0, 1), (1, 0, -1), (-1, 0, -1), (0, 1, 1), (0, -1, 1), (0, 1, -1),
      (0, -1, -1)]
_INV = [_C.index((-x, -y, -z)) for x, y, z in _C]
_W = [1 / 3 if c == (0, 0, 0) else (1 / 18 if sum(map(abs, c)) == 1 else 1 / 36) for c in _C]


def _at(f, c):
    """f at r + c, for f (..., lz, ly, lx)."""
    return torch.roll(f, (-c[2], -c[1], -c[0]), (-3, -2, -1))


def _exact_flow(solid, tau, F, steps):
    """D3Q19 BGK with Guo forcing and half-way bounce-back in torch's FP64:
    rest for three steps (the force is switched on by the first convergence,
    at step 3), the force from step 4.  solid (B, lz, ly, lx)."""
    fluid = (~solid).to(torch.float64)
    col = lambda v: torch.tensor(v, dtype=torch.float64, device="cuda").reshape(-1, 1, 1, 1, 1)  # noqa: E731
    w, cx, cy, cz = col(_W), *(col([float(c[a]) for c in _C]) for a in range(3))
    from_solid = [_at(solid, _C[_INV[q]]) for q in range(19)]  # r - c is solid
    n = w * fluid
    rho, j = fluid.clone(), torch.zeros((3,) + tuple(solid.shape), dtype=torch.float64, device="cuda")
    l2 = []
    for t in range(1, steps + 1):
        fn = F if t > 3 else [0.0, 0.0, 0.0]    # the force of step t's collision
        safe = torch.where(solid, 1.0, rho)
        u = j / safe
        cj = cx * j[0] + cy * j[1] + cz * j[2]
        cu = cx * u[0] + cy * u[1] + cz * u[2]
        cF = cx * fn[0] + cy * fn[1] + cz * fn[2]
        ju, uF = (j * u).sum(0), u[0] * fn[0] + u[1] * fn[1] + u[2] * fn[2]
        neq = w * (rho + 3.0 * cj + 4.5 * (cj * cu - ju / 3.0))
        n = (1 - 1 / tau) * n + neq / tau + (1 - 1 / (2 * tau)) * w * (3.0 * (cF - uF) + 9.0 * cu * cF)
        n = n * fluid
        n = torch.stack([torch.where(from_solid[q], n[_INV[q]], _at(n[q], _C[_INV[q]])) for q in range(19)]) * fluid
        rho = n.sum(0)
        new = torch.stack([(n * cx).sum(0) + fn[0] / 2, (n * cy).sum(0) + fn[1] / 2, (n * cz).sum(0) + fn[2] / 2])
        new = new * fluid
        l2.append((new - j).abs().amax(dim=(0, 2, 3, 4)))
        j = new
    return n, rho, j, torch.stack(l2)


def _exact_tracer(solid, rho, j, F, ka, kd, steps, want_p):
    """Moment propagation of one tracer per lattice in torch's FP64; ka, kd
    are (B,) tensors.  solid (B, lz, ly, lx)."""
    fluid = ~solid
    safe = torch.where(solid, 1.0, rho)
    u = [torch.where(solid, 0.0, (j[a] + F[a]) / safe) for a in range(3)]
    lam = 4.0 * DB * 3.0
    B = solid.shape[0]
    inter = torch.zeros_like(solid)
    rem, us = fluid.to(torch.float64), torch.zeros_like(j)
    into, v0_dir = [], torch.zeros((3, B), dtype=torch.float64, device="cuda")
    p1 = torch.zeros_like(j)
    for q in range(1, 19):
        c = _C[q]
        s = _W[q] * (3.0 * (c[0] * u[0] + c[1] * u[1] + c[2] * u[2]) + lam / 2)
        inter |= fluid & _at(solid, c)
        s_out = torch.where(fluid & _at(fluid, c), s, 0.0)
        rem = rem - s_out
        c_in = _C[_INV[q]]
        s_in = _W[q] * (3.0 * (c_in[0] * u[0] + c_in[1] * u[1] + c_in[2] * u[2]) + lam / 2)
        s_in = torch.where(fluid & _at(fluid, c), _at(s_in, c), 0.0)
        into.append(s_in)
        for a in range(3):
            if c[a]:
                us[a] += c[a] * s_out
                v0_dir[a] += s_out.sum(dim=(1, 2, 3))
                p1[a] -= c[a] * s_in
    nf, ni = fluid.sum(dim=(1, 2, 3)).double(), inter.sum(dim=(1, 2, 3)).double()
    bw = 1.0 / (nf + ka / kd * ni)
    wall = inter.to(torch.float64)
    kab, kdb = ka.reshape(-1, 1, 1, 1) * wall, kd.reshape(-1, 1, 1, 1) * wall
    P, Pa, v0 = p1 * bw.reshape(-1, 1, 1, 1), torch.zeros_like(p1), v0_dir * bw
    vacf = []
    for _ in range(steps):
        vacf.append((P * us).sum(dim=(2, 3, 4)))
        new = (rem - kab) * P + kdb * Pa
        for q in range(1, 19):
            new.addcmul_(_at(P, _C[q]), into[q - 1].expand_as(P))
        Pa = (1 - kdb) * Pa + kab * P
        P = new
    vacf = torch.stack(vacf)  # (steps, 3, B)
    d = v0 / 2 + vacf.sum(0)
    out = {"vacf0": v0.T, "vacf": vacf.permute(2, 0, 1), "deff": d.T}
    if want_p:
        out["P"], out["Pa"] = (x.permute(1, 2, 3, 4, 0).reshape(B, -1) for x in (P, Pa * wall))
    return out


def _vec(x):
    return torch.tensor(x, dtype=torch.float64, device="cuda")


def _exact_batch(c, seed):
    reqs = _requests(c, seed)
    deff, vacf = [None] * len(reqs), [None] * len(reqs)
    # lattices of one size and force direction run together in torch, each with its own force
    groups = {}
    for k, r in enumerate(reqs):
        groups.setdefault((r[0], r[1]), []).append(k)
    for ks in groups.values():
        solid = torch.stack([reqs[k][2] for k in ks])
        F = [_vec([reqs[k][3][a] for k in ks]).reshape(-1, 1, 1, 1) for a in range(3)]
        _, rho, j, _ = _exact_flow(solid, c["tau"], F, c["lb_steps"])
        t = _exact_tracer(solid, rho, j, F, _vec([reqs[k][4] for k in ks]), _vec([reqs[k][5] for k in ks]),
                          c["mp_steps"], False)
        for i, k in enumerate(ks):
            deff[k], vacf[k] = t["deff"][i], torch.cat([t["vacf0"][i][None], t["vacf"][i]])
    return {"deff": torch.stack(deff), "vacf": torch.stack(vacf)}


def exact(case, seed):
    c = case
    if c["path"] == "batch":
        return _exact_batch(c, seed)
    solid, F, ka, kd = _inputs(c, seed)
    solid = solid[None]
    n, rho, j, l2 = _exact_flow(solid, c["tau"], F, c["lb_steps"] or FLOW_STEPS)
    flow = {"l2err": l2.reshape(-1) if c["prec"] == "fp64" else None, "rho": rho.reshape(-1), "j": j.reshape(3, -1)}
    if c["path"] == "flow":
        return flow
    ts = [_exact_tracer(solid, rho, j, F, _vec([a]), _vec([d]), c["mp_steps"], c["path"] == "solve")
          for a, d in zip(ka, kd)]
    if c["path"] == "tracers":
        return {"vacf0": torch.stack([t["vacf0"][0] for t in ts]),
                "vacf": torch.stack([t["vacf"][0] for t in ts], 1), "deff": torch.stack([t["deff"][0] for t in ts])}
    out = {**flow, **{k: v[0] for k, v in ts[0].items()}}
    if c["path"] == "program":
        out["n"] = n.reshape(-1)
    return out
