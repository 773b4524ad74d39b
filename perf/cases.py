"""Performance cases of the MHD update: what a user's program has the library do, through
its public entry points (``athena_amd.gpu`` and the C ABI it mirrors).

Kinds of case:

* ``evolve``: one uniform mesh advanced ``cycles`` VL2 cycles and its conserved state (u and
  the face field of every MeshBlock, ghosts included) read back to the host, as a run that
  dumps every ``cycles`` cycles does.  Newtonian or special-relativistic, donor cell / PLM /
  PPM, HLLD / HLLE, periodic or outflow faces, launched eagerly or as HIP graphs.
* ``ensemble``: independent blast waves of uneven sizes advanced together.
* ``refined``: the statically refined linear-wave mesh.
* ``recover``: batched special-relativistic primitive recovery over device arrays.
* ``block``: the per-MeshBlock functions of one VL2 stage over arrays the caller owns.

``exact`` integrates the same equations on one global grid in plain torch, in 64 bits.
"""
import math

import numpy as np
import torch

from athena_amd import gpu, ml
from athena_amd.mesh import DEFAULT_FLOOR, MeshDesc, refined
from athena_amd.pgen.blast import Blast, blast_mesh
from athena_amd.pgen.linear_wave import LinearWave, linear_wave_mesh
from athena_amd.pgen.sr import ShearLayer
from athena_amd.pgen.turbulence import Turbulence

# The five refined regions of the reference's refined linear-wave input.
REGIONS = [((0.7, 0.1, 0.3), (0.8, 0.3, 0.4), 1), ((0.4, 0.8, 1.2), (0.6, 0.9, 1.4), 1),
           ((2.0, 0.5, 0.6), (2.4, 0.6, 0.8), 1), ((1.2, 0.4, 0.2), (1.6, 0.8, 0.4), 1),
           ((1.6, 1.2, 1.1), (2.2, 1.4, 1.3), 1)]


def _evolve(problem, nx, bnx, cycles, xorder=2, ng=2, rsolver="hlld", graph=False,
            bc="periodic"):
    return {"kind": "evolve", "problem": problem, "nx1": nx[0], "nx2": nx[1], "nx3": nx[2],
            "bnx1": bnx[0], "bnx2": bnx[1], "bnx3": bnx[2], "cycles": cycles,
            "xorder": xorder, "ng": ng, "rsolver": rsolver, "graph": graph, "bc": bc}


def listed():
    c = [
        # the regression suite's linear wave: one small MeshBlock, launch latency counts
        dict(_evolve("wave", (32, 16, 16), (32, 16, 16), 20), name="wave32"),
        # the linear-wave parity run: 64^3, a few MeshBlocks
        dict(_evolve("wave", (64, 64, 64), (32, 32, 32), 20, graph=True), name="wave64"),
        # decaying turbulence at an ordinary size
        dict(_evolve("turbulence", (128,) * 3, (32,) * 3, 100, graph=True), name="turb128"),
        # the headline workload: 256^3 as 512 MeshBlocks
        dict(_evolve("turbulence", (256,) * 3, (32,) * 3, 60, graph=True), name="turb256"),
        # third-order reconstruction on MeshBlocks of uneven edges, launched eagerly
        dict(_evolve("turbulence", (120,) * 3, (40, 30, 24), 50, xorder=3, ng=3),
             name="ppm120"),
        # a blast wave in an open box, HLLE, larger MeshBlocks
        dict(_evolve("blast", (96,) * 3, (48,) * 3, 100, rsolver="hlle", bc="outflow"),
             name="blast96"),
        # relativistic shear layer: PPM, HLLE, iterative primitive recovery
        dict(_evolve("shear", (128,) * 3, (32,) * 3, 40, xorder=3, ng=3, rsolver="hlle",
                     graph=True), name="shear128"),
        # an ensemble study: blast waves of uneven sizes advanced together
        {"kind": "ensemble", "members": 12, "largest": 96, "cycles": 40, "name": "ensemble12"},
        # static refinement: the regression mesh, two levels
        {"kind": "refined", "nx1": 128, "bn": 16, "cycles": 40, "name": "refined128"},
        # primitive recovery of 128^3 states from a cold start
        {"kind": "recover", "n": 128 ** 3, "mode": 0, "name": "recover128"},
        # the same with the learned guess, a smaller ragged batch
        {"kind": "recover", "n": 250007, "mode": 2, "name": "recover_learned"},
        # per-MeshBlock functions as another program's task list calls them
        {"kind": "block", "nx1": 64, "nx2": 64, "nx3": 64, "order": 2, "ng": 2,
         "rsolver": "hlld", "name": "block64"},
    ]
    return c


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["evolve"] * 5 + ["shear"] * 2 + ["ensemble", "refined", "recover",
                                                       "recover", "block"])
    if kind in ("evolve", "shear"):
        edge = _log_int(rng, 16, 176 if kind == "evolve" else 128)   # cells per direction
        nb = max(1, int(round(edge / rng.uniform(12, 56))))
        bn = max(4, edge // nb)
        xorder = rng.choice([1, 2, 2, 2, 3])
        cycles = max(4, min(100, int(2.5e8 / float(bn * nb) ** 3)))
        if kind == "shear":
            n = bn * nb
            return _evolve("shear", (n,) * 3, (bn,) * 3, max(4, cycles // 3),
                           xorder=rng.choice([2, 3]), ng=3,
                           rsolver=rng.choice(["hlle", "hlle", "hlld"]),
                           graph=rng.random() < 0.5)
        # a blast keeps to DC and PLM: PPM's limiter jumps on the rounding noise of its
        # uniform surroundings, so that no tolerance could be stated
        problem = rng.choice(["turbulence", "turbulence", "wave"] +
                             ([] if xorder == 3 else ["blast"]))
        n = bn * nb
        if problem == "turbulence":
            nx, bnx = (n,) * 3, (bn,) * 3
        else:   # uneven edges too
            b2, b3 = rng.choice([bn, max(4, bn - 3)]), rng.choice([bn, max(4, bn - 5)])
            nx, bnx = (n, b2 * nb, b3 * nb), (bn, b2, b3)
        return _evolve(problem, nx, bnx, cycles, xorder=xorder, ng=3 if xorder == 3 else 2,
                       rsolver=rng.choice(["hlld", "hlld", "hlle"]),
                       graph=rng.random() < 0.5,
                       bc="outflow" if problem == "blast" and rng.random() < 0.5 else "periodic")
    if kind == "ensemble":
        return {"kind": "ensemble", "members": rng.randint(3, 14),
                "largest": rng.choice([48, 64, 96]), "cycles": rng.randint(10, 40)}
    if kind == "refined":
        return {"kind": "refined", "nx1": rng.choice([64, 96, 128]),
                "bn": rng.choice([8, 16]), "cycles": rng.randint(10, 40)}
    if kind == "recover":
        return {"kind": "recover", "n": _log_int(rng, 1000, 4000000),
                "mode": rng.choice([0, 0, 1, 2])}
    order = rng.choice([1, 2, 2, 3])
    return {"kind": "block", "nx1": rng.randint(16, 100), "nx2": rng.randint(16, 80),
            "nx3": rng.randint(16, 80), "order": order, "ng": 3 if order == 3 else 2,
            "rsolver": rng.choice(["hlld", "hlld", "hlle"])}


# ---------------------------------------------------------------------------------------
# Meshes and their initial conditions

def _mesh(case):
    nx = (case["nx1"], case["nx2"], case["nx3"])
    bnx = (case["bnx1"], case["bnx2"], case["bnx3"])
    kw = dict(nx=nx, bnx=bnx, xorder=case["xorder"], ng=case["ng"], rsolver=case["rsolver"],
              bc=(case["bc"],) * 6, cfl=0.3, gamma=5.0 / 3.0)
    p = case["problem"]
    if p == "wave":
        return MeshDesc(xmin=(0.0,) * 3, xmax=(3.0, 1.5, 1.5), **kw)
    if p == "blast":
        return MeshDesc(xmin=(-1.0,) * 3, xmax=(1.0,) * 3, **kw)
    if p == "shear":
        return MeshDesc(xmin=(-0.5,) * 3, xmax=(0.5,) * 3, relativistic=True,
                        **dict(kw, gamma=4.0 / 3.0))
    return MeshDesc(xmin=(-0.5,) * 3, xmax=(0.5,) * 3, **kw)


def _problem(case, m, seed):
    rng = np.random.default_rng(seed)
    p = case["problem"]
    if p == "wave":
        return LinearWave(m, wave_flag=int(rng.integers(0, 7)),
                          amp=float(10.0 ** rng.uniform(-6, -3)),
                          vflow=float(rng.uniform(0.0, 0.5)))
    if p == "blast":
        return Blast(m, prat=float(10.0 ** rng.uniform(1, 2.5)), radius=0.25,
                     b0=float(rng.uniform(0.1, 1.0)), bdir=rng.normal(size=3),
                     center=tuple(rng.uniform(-0.2, 0.2, 3)))
    if p == "shear":
        return ShearLayer(m, seed=seed, width=0.05)
    return Turbulence(m, seed=seed)


def _ensemble_members(case, seed):
    """The members' sizes are part of the case; their waves come from the seed."""
    edges = [e for e in (32, 48, 64, 96) if e <= case["largest"]]
    rng = np.random.default_rng(seed)
    out = []
    for q in range(case["members"]):
        n = edges[::-1][q % len(edges)]
        m = blast_mesh(n, 32 if n % 32 == 0 else 16)
        out.append((m, Blast(m, prat=float(np.exp(rng.uniform(np.log(10.0), np.log(1000.0)))),
                             b0=float(rng.uniform(0.1, 1.0)), bdir=rng.normal(size=3))))
    return out


def _refined_mesh(case):
    n = case["nx1"]
    return refined(linear_wave_mesh(n, 0, bnx=(case["bn"],) * 3), REGIONS)


KEYS = ("u", "b1", "b2", "b3")


class _Dump:
    """Host (pinned) arrays the conserved state of a mesh is read back into: u of every
    MeshBlock, then the face fields, ghosts included."""

    def __init__(self, mesh):
        self.mesh = mesh
        pin = torch.cuda.is_available()
        self.out = {k: torch.empty((mesh.m.nblocks,) + tuple(mesh.m.shape(k)),
                                   dtype=torch.float64, pin_memory=pin) for k in KEYS}
        self.args = []
        for k in KEYS:
            t = self.out[k]
            for g in range(mesh.m.nblocks):
                p = gpu.ctypes.cast(t[g].data_ptr(), gpu.ctypes.POINTER(gpu.ctypes.c_double))
                self.args.append((g, gpu.ATH[k], p))

    def read(self):
        get, h = gpu.load().ath_gpu_get_block, self.mesh.h
        for g, code, p in self.args:
            if get(h, g, code, p):
                raise gpu.AthGpuError(gpu.load().ath_gpu_last_error().decode())
        return self.out


def _device_mesh(m, problem):
    d = gpu.GpuMesh(m)
    keys = KEYS + (("w", "w1") if m.relativistic else ())
    for g in range(m.nblocks):
        b = problem.block(g)
        for k in keys:
            d.set(g, k, b[k])
    d.initialize()
    return d


def prepare(case, seed):
    kind = case["kind"]
    if kind == "evolve":
        m = _mesh(case)
        d = _device_mesh(m, _problem(case, m, seed))
        d.set_graph(case["graph"])
        return {"case": case, "mesh": d, "dump": _Dump(d)}
    if kind == "ensemble":
        meshes = [_device_mesh(m, p) for m, p in _ensemble_members(case, seed)]
        return {"case": case, "meshes": meshes, "ens": gpu.Ensemble(meshes),
                "dumps": [_Dump(d) for d in meshes]}
    if kind == "refined":
        m = _refined_mesh(case)
        rng = np.random.default_rng(seed)
        wave = LinearWave(m, wave_flag=int(rng.integers(0, 7)),
                          amp=float(10.0 ** rng.uniform(-6, -3)))
        d = _device_mesh(m, wave)
        d.set_graph(True)
        return {"case": case, "mesh": d, "dump": _Dump(d)}
    if kind == "recover":
        cons, bcc, _ = ml.conserved_batch(case["n"], seed)
        dev = torch.device("cuda:0")
        c = torch.from_numpy(cons).to(dev)
        return {"case": case, "cons": c, "prim": torch.empty_like(c),
                "bcc": torch.from_numpy(bcc).to(dev),
                "net": ml.load_mlp() if case["mode"] == 2 else None}
    return _prepare_block(case, seed)


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind in ("evolve", "refined"):
        s["mesh"].run(case["cycles"])
        return dict(s["dump"].read(), clock=list(s["mesh"].state()))
    if kind == "ensemble":
        s["ens"].run(case["cycles"])
        return [dict(d.read()) for d in s["dumps"]]
    if kind == "recover":
        s["prim"].zero_()          # cold: no previous primitives
        gpu.sr_con2prim_device(case["mode"], case["n"], s["cons"].data_ptr(),
                               s["prim"].data_ptr(), s["bcc"].data_ptr(), ml.GAMMA_AD,
                               DEFAULT_FLOOR, DEFAULT_FLOOR, mlp=s["net"])
        return {"cons": s["cons"], "prim": s["prim"]}
    return _run_block(s)


# ---------------------------------------------------------------------------------------
# One VL2 stage of one MeshBlock over caller-owned arrays

def _block_mesh(case):
    nx = (case["nx1"], case["nx2"], case["nx3"])
    return MeshDesc(nx=nx, bnx=nx, xmin=(-0.5,) * 3, xmax=(0.5,) * 3, ng=case["ng"],
                    rsolver=case["rsolver"], xorder=case["order"], gamma=5.0 / 3.0, cfl=0.3)


def _block_state(case, seed, dev):
    """Primitives, faces and cell-centred field of one MeshBlock with its ghosts: a smooth
    large-scale flow with 5 % cell noise; the faces are uniform plus noise."""
    m = _block_mesh(case)
    g = torch.Generator(device="cpu").manual_seed(seed)
    c1, c2, c3 = m.nc

    def noise(*shape):
        return torch.randn(shape, generator=g, dtype=torch.float64)

    x = [torch.arange(n, dtype=torch.float64) / n * 2 * math.pi for n in (c1, c2, c3)]
    ph = torch.rand(5, 3, generator=g, dtype=torch.float64) * 2 * math.pi
    w = torch.stack([torch.sin(x[2] + ph[v, 2])[:, None, None] *
                     torch.sin(x[1] + ph[v, 1])[None, :, None] *
                     torch.sin(2 * x[0] + ph[v, 0])[None, None, :] for v in range(5)])
    w = w + 0.05 * noise(5, c3, c2, c1)
    w[0] = 1.0 + 0.3 * torch.tanh(w[0])
    w[4] = 1.0 + 0.4 * torch.tanh(w[4])
    f = [0.3 + 0.1 * noise(c3, c2, c1 + 1), 0.2 + 0.1 * noise(c3, c2 + 1, c1),
         -0.1 + 0.1 * noise(c3 + 1, c2, c1)]
    bcc = torch.stack([0.5 * f[0][:, :, :-1] + 0.5 * f[0][:, :, 1:],
                       0.5 * f[1][:, :-1] + 0.5 * f[1][:, 1:],
                       0.5 * f[2][:-1] + 0.5 * f[2][1:]])
    ke = 0.5 * w[0] * (w[1] ** 2 + w[2] ** 2 + w[3] ** 2)
    e = w[4] / (m.gamma - 1) + ke + 0.5 * (bcc ** 2).sum(0)
    u = torch.stack([w[0], w[0] * w[1], w[0] * w[2], w[0] * w[3], e])
    dt = 0.05 / max(m.nx)
    return m, dt, [t.contiguous().to(dev) for t in (w, bcc, u)], [t.to(dev) for t in f]


def _prepare_block(case, seed):
    dev = torch.device("cuda:0")
    m, dt, (w, bcc, u), f = _block_state(case, seed, dev)
    c1, c2, c3 = m.nc
    face = [(c3, c2, c1 + 1), (c3, c2 + 1, c1), (c3 + 1, c2, c1)]
    edge = [(c3 + 1, c2 + 1, c1), (c3 + 1, c2, c1 + 1), (c3, c2 + 1, c1 + 1)]

    def zeros(*shape):
        return torch.zeros(shape, dtype=torch.float64, device=dev)

    r = {}
    for q in range(3):
        r["flux%d" % (q + 1)] = zeros(5, *face[q])
        r["wght%d" % (q + 1)] = zeros(*face[q])
        r["e%d" % (q + 1)] = zeros(*edge[q])
    for n, q in (("e3_x1f", 0), ("e2_x1f", 0), ("e1_x2f", 1), ("e3_x2f", 1), ("e2_x3f", 2),
                 ("e1_x3f", 2)):
        r[n] = zeros(*face[q])
    return {"case": case, "dt": dt, "w": w, "bcc": bcc, "f": f, "u0": u, "regs": r, "m": m,
            "addr": {k: t.data_ptr() for k, t in r.items()},
            "blk": gpu.Block(m), "u": u.clone(), "b": [t.clone() for t in f],
            "w_out": w.clone(), "bcc_out": bcc.clone(), "new_dt": zeros(1)}


def _run_block(s):
    blk, a, m, dt = s["blk"], s["addr"], s["m"], s["dt"]
    w, bcc = s["w"].data_ptr(), s["bcc"].data_ptr()
    b = [t.data_ptr() for t in s["f"]]
    blk.calculate_fluxes(w, b[0], b[1], b[2], bcc, s["case"]["order"], dt, a)
    blk.compute_corner_e(w, bcc, a)
    s["u"].copy_(s["u0"])          # the caller's weighted average into the output register
    for q in range(3):
        s["b"][q].copy_(s["f"][q])
    o = [t.data_ptr() for t in s["b"]]
    blk.ct(dt, a, o[0], o[1], o[2])
    blk.add_flux_divergence(dt, a, s["u"].data_ptr())
    n = m.nc
    blk.cons2prim(s["u"].data_ptr(), w, o[0], o[1], o[2], s["w_out"].data_ptr(),
                  s["bcc_out"].data_ptr(), (0, n[0] - 1, 0, n[1] - 1, 0, n[2] - 1))
    blk.new_dt_noalloc(s["w_out"].data_ptr(), s["bcc_out"].data_ptr(), o[0], o[1], o[2],
                       s["new_dt"].data_ptr())
    return {"u": s["u"], "b": s["b"], "w": s["w_out"], "bcc": s["bcc_out"],
            "dt": s["new_dt"], "e": [s["regs"]["e%d" % q] for q in (1, 2, 3)],
            "flux": [s["regs"]["flux%d" % q] for q in (1, 2, 3)]}


# ---------------------------------------------------------------------------------------
# Work and tolerances

def _cells(case):
    kind = case["kind"]
    if kind == "evolve":
        return case["nx1"] * case["nx2"] * case["nx3"]
    if kind == "ensemble":
        return sum(m.nx[0] ** 3 for m, _ in _ensemble_members(case, 0))
    if kind == "refined":
        return _refined_mesh(case).nblocks * case["bn"] ** 3
    if kind == "recover":
        return case["n"]
    return case["nx1"] * case["nx2"] * case["nx3"]


def work(case):
    """Bytes: per VL2 cycle and cell 67 doubles (stage 1 reads U, B, W and Bcc and writes
    their half-step values, stage 2 reads U, B and the half-step values and writes the new
    ones), plus the state read back; a recovery 19 doubles (cons, prim and bcc in, cons and
    prim out, less the cold seed); a MeshBlock stage its inputs and outputs once.  FLOPs: three
    Riemann solves per cell and stage with their reconstruction, the corner EMFs, the update
    and the recovery, counted from their formulas."""
    n = float(_cells(case))
    if case["kind"] == "recover":
        return {"bytes": n * 8 * 13, "flops": n * 600}
    if case["kind"] == "block":
        return {"bytes": n * 8 * (8 + 3 + 5 + 5 + 3 + 8 + 15 + 3), "flops": n * 2400}
    stage = {1: 1500, 2: 2400, 3: 4200}[case.get("xorder", 2)]
    per = 1500 + stage
    return {"bytes": n * (536.0 * case["cycles"] + 64.0), "flops": n * per * case["cycles"]}


def tolerance(case):
    """FP64 throughout; about four times what the library is away from exact().  Newtonian
    meshes: up to 3e-15 over 20 to 100 cycles, with room for longer drawn runs; one stage of
    one MeshBlock: up to 3e-16.  The relativistic recovery stops at an absolute 1e-12 in the
    gas pressure, which the batched states hold down to 1e-5: 2e-11 to 5e-11, and 2e-10 in the
    shear layer's small transverse field."""
    if case["kind"] == "block":
        return {"rel": 1.2e-15, "max": 1e-13}
    if case["kind"] == "recover":
        return {"rel": 2e-10}
    if case.get("problem") == "shear":
        return {"rel": 8e-10}
    return {"rel": 2e-14, "max": 1e-11}


# ---------------------------------------------------------------------------------------
# The same equations on one global grid in plain torch, 64 bits

def _sq(x):
    return x * x


def _vl(qm, q0, qp):
    a, b = q0 - qm, qp - q0
    p = a * b
    s = torch.where(p > 0, a + b, torch.ones_like(p))
    return torch.where(p > 0, 2 * p / s, torch.zeros_like(p))


def _ppm_edges(q):
    """Colella & Sekora (2008) limited edge values (left, right) of the middle cells of q
    along its last axis (two cells lost on each side)."""
    C = 1.25
    m2, m1, c, p1, p2 = (q[..., i:q.shape[-1] - 4 + i] for i in range(5))
    sg = lambda x: torch.where(x < 0, -torch.ones_like(x), torch.ones_like(x))  # noqa: E731
    d2m, d2, d2p = m2 + c - 2 * m1, m1 + p1 - 2 * c, c + p2 - 2 * p1

    def iface(a2, a1, b1, b2, da, db):
        f = 0.5 * (a1 + b1) + (0.5 * (b1 - a2) - 0.5 * (b2 - a1)) / 6
        d = 3 * (a1 + b1 - 2 * f)
        lim = torch.where((sg(d) == sg(da)) & (sg(d) == sg(db)),
                          sg(d) * torch.minimum(C * da.abs(), torch.minimum(C * db.abs(),
                                                                            d.abs())),
                          torch.zeros_like(d))
        return torch.where((f - a1) * (b1 - f) < 0, 0.5 * (a1 + b1) - lim / 6, f)

    lo = iface(m2, m1, c, p1, d2m, d2)
    hi = iface(m1, c, p1, p2, d2, d2p)
    d2f = 6 * (lo + hi - 2 * c)
    dm, dp = c - lo, hi - c
    same = (sg(d2m) == sg(d2)) & (sg(d2m) == sg(d2p)) & (sg(d2m) == sg(d2f))
    lim = torch.where(same, sg(d2f) * torch.minimum(
        torch.minimum(C * d2m.abs(), C * d2.abs()), torch.minimum(C * d2p.abs(), d2f.abs())),
        torch.zeros_like(c))
    big = torch.stack([m1.abs(), m2.abs(), c.abs(), p1.abs(), p2.abs()]).amax(0)
    ok = d2f.abs() > 1e-12 * big
    rho = torch.where(ok, lim / torch.where(ok, d2f, torch.ones_like(d2f)),
                      torch.zeros_like(c))
    ext = (dm * dp <= 0) | ((p1 - c) * (c - m1) <= 0)
    flat = rho <= 1 - 1e-12
    lo2 = torch.where(ext, torch.where(flat, c - rho * dm, lo),
                      torch.where(dm.abs() >= 2 * dp.abs(), c - 2 * dp, lo))
    hi2 = torch.where(ext, torch.where(flat, c + rho * dp, hi),
                      torch.where(dp.abs() >= 2 * dm.abs(), c + 2 * dm, hi))
    return lo2, hi2


def _states(q, g, order):
    """Left and right states at the n + 1 faces of the active range along the last axis."""
    n = q.shape[-1] - 2 * g
    if order == 1:
        return q[..., g - 1:g + n], q[..., g:g + n + 1]
    if order == 2:
        d = _vl(q[..., :-2], q[..., 1:-1], q[..., 2:])      # of cells 1 ..
        lo, hi = q[..., 1:-1] - 0.5 * d, q[..., 1:-1] + 0.5 * d
        return hi[..., g - 2:g - 1 + n], lo[..., g - 1:g + n]
    lo, hi = _ppm_edges(q)                                    # of cells 2 ..
    return hi[..., g - 3:g - 2 + n], lo[..., g - 2:g - 1 + n]


def _fast(w, bx, gam):
    a, v, t = gam * w[4], bx * bx, _sq(w[5]) + _sq(w[6])
    return torch.sqrt(0.5 * (v + t + a + torch.sqrt(_sq(v + t - a) + 4 * a * t)) / w[0])


def _mhd_side(w, bx, gam):
    d, vx, vy, vz, p, by, bz = w
    pb = 0.5 * (bx * bx + by * by + bz * bz)
    e = p / (gam - 1) + 0.5 * d * (vx * vx + vy * vy + vz * vz) + pb
    pt = p + pb
    vb = vx * bx + vy * by + vz * bz
    u = torch.stack([d, d * vx, d * vy, d * vz, e, by, bz])
    f = torch.stack([d * vx, d * vx * vx + pt - bx * bx, d * vy * vx - bx * by,
                     d * vz * vx - bx * bz, (e + pt) * vx - bx * vb, by * vx - bx * vy,
                     bz * vx - bx * vz])
    return u, f, pt


def _hlle(wl, wr, bx, gam):
    g1 = gam - 1
    ul, fl, ptl = _mhd_side(wl, bx, gam)
    ur, fr, ptr = _mhd_side(wr, bx, gam)
    sl, sr = torch.sqrt(wl[0]), torch.sqrt(wr[0])
    s = 1 / (sl + sr)
    d = sl * sr
    v = [(sl * wl[k] + sr * wr[k]) * s for k in (1, 2, 3)]
    b = [(sr * wl[k] + sl * wr[k]) * s for k in (5, 6)]
    x = 0.5 * (_sq(wl[5] - wr[5]) + _sq(wl[6] - wr[6])) / _sq(sl + sr)
    y = 0.5 * (wl[0] + wr[0]) / d
    h = ((ul[4] + ptl) / sl + (ur[4] + ptr) / sr) * s
    bt = b[0] * b[0] + b[1] * b[1]
    va = bx * bx / d
    a2 = (g1 * (h - va - bt / d - 0.5 * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2)) -
          (g1 - 1) * x).clamp(min=0)
    ct = (g1 - (g1 - 1) * y) * bt / d
    cf = torch.sqrt(0.5 * (va + ct + a2 + torch.sqrt(_sq(va + ct - a2) + 4 * a2 * ct)))
    lo = torch.minimum(v[0] - cf, wl[1] - _fast(wl, bx, gam)).clamp(max=0)
    hi = torch.maximum(v[0] + cf, wr[1] + _fast(wr, bx, gam)).clamp(min=0)
    return (hi * fl - lo * fr + hi * lo * (ur - ul)) / (hi - lo)


def _hlld(wl, wr, bx, gam):
    """Miyoshi & Kusano (2005)."""
    ul, fl, ptl = _mhd_side(wl, bx, gam)
    ur, fr, ptr = _mhd_side(wr, bx, gam)
    cl, cr = _fast(wl, bx, gam), _fast(wr, bx, gam)
    s0, s4 = torch.minimum(wl[1] - cl, wr[1] - cr), torch.maximum(wl[1] + cl, wr[1] + cr)
    dl, dr = s0 - wl[1], s4 - wr[1]
    s2 = (dr * ur[1] - dl * ul[1] + ptl - ptr) / (dr * ur[0] - dl * ul[0])
    pts = 0.5 * (ptl + ul[0] * dl * (s2 - wl[1]) + ptr + ur[0] * dr * (s2 - wr[1]))

    def star(w, u, pt, sd, s):
        sm = s - s2
        d = u[0] * sd / sm
        den = u[0] * sd * sm - bx * bx
        deg = den.abs() < 1e-4 * pts
        den = torch.where(deg, torch.ones_like(den), den)
        t = torch.where(deg, torch.zeros_like(den), bx * (sd - sm) / den)
        r = torch.where(deg, torch.ones_like(den), (u[0] * sd * sd - bx * bx) / den)
        vy, vz, by, bz = w[2] - w[5] * t, w[3] - w[6] * t, w[5] * r, w[6] * r
        vb = s2 * bx + vy * by + vz * bz
        e = (sd * u[4] - pt * w[1] + pts * s2 +
             bx * (w[1] * bx + w[2] * w[5] + w[3] * w[6] - vb)) / sm
        return torch.stack([d, d * s2, d * vy, d * vz, e, by, bz]), vb

    a, vba = star(wl, ul, ptl, dl, s0)
    c, vbc = star(wr, ur, ptr, dr, s4)
    ra, rc = torch.sqrt(a[0]), torch.sqrt(c[0])
    s1, s3 = s2 - bx.abs() / ra, s2 + bx.abs() / rc
    inv = 1 / (ra + rc)
    sg = torch.where(bx > 0, torch.ones_like(bx), -torch.ones_like(bx))
    vy = inv * (ra * a[2] / a[0] + rc * c[2] / c[0] + sg * (c[5] - a[5]))
    vz = inv * (ra * a[3] / a[0] + rc * c[3] / c[0] + sg * (c[6] - a[6]))
    by = inv * (ra * c[5] + rc * a[5] + sg * ra * rc * (c[2] / c[0] - a[2] / a[0]))
    bz = inv * (ra * c[6] + rc * a[6] + sg * ra * rc * (c[3] / c[0] - a[3] / a[0]))
    vb = s2 * bx + vy * by + vz * bz
    aa = torch.stack([a[0], a[1], a[0] * vy, a[0] * vz, a[4] - ra * sg * (vba - vb), by, bz])
    cc = torch.stack([c[0], c[1], c[0] * vy, c[0] * vz, c[4] + rc * sg * (vbc - vb), by, bz])
    fa, fc = fl + s0 * (a - ul), fr + s4 * (c - ur)
    f = torch.where(s2 >= 0, fa + s1 * (aa - a), fc + s3 * (cc - c))
    f = torch.where(s3 <= 0, fc, torch.where(s1 >= 0, fa, f))
    return torch.where(s0 >= 0, fl, torch.where(s4 <= 0, fr, f))


def _sr_hlle(wl, wr, bx, gam):
    def side(w):
        d, x, y, z, p, by, bz = w
        u0 = torch.sqrt(1 + x * x + y * y + z * z)
        b0 = bx * x + by * y + bz * z
        b1, b2, b3 = (bx + b0 * x) / u0, (by + b0 * y) / u0, (bz + b0 * z) / u0
        bb = b1 * b1 + b2 * b2 + b3 * b3 - b0 * b0
        wg = d + gam / (gam - 1) * p
        wt, pt = wg + bb, p + 0.5 * bb
        u = torch.stack([d * u0, wt * u0 * x - b0 * b1, wt * u0 * y - b0 * b2,
                         wt * u0 * z - b0 * b3, wt * u0 * u0 - b0 * b0 - pt, by, bz])
        f = torch.stack([d * x, wt * x * x - b1 * b1 + pt, wt * x * y - b1 * b2,
                         wt * x * z - b1 * b3, wt * u0 * x - b0 * b1, b2 * x - b1 * y,
                         b3 * x - b1 * z])
        cs, va = gam * p / wg, bb / wt
        cm = cs + va - cs * va
        qa = u0 * u0 - (u0 * u0 - 1) * cm
        qb = -2 * u0 * x * (1 - cm)
        qc = x * x - (1 + x * x) * cm
        r = torch.sqrt((qb * qb - 4 * qa * qc).clamp(min=0))
        return u, f, (-qb - r) / (2 * qa), (-qb + r) / (2 * qa)

    ul, fl, l0, l1 = side(wl)
    ur, fr, r0, r1 = side(wr)
    lo, hi = torch.minimum(l0, r0).clamp(max=0), torch.maximum(l1, r1).clamp(min=0)
    return (hi * fl - lo * fr + lo * hi * (ur - ul)) / (hi - lo)


def _sr_primitives(u, b, gam):
    """Gas pressure root of the energy equation in W = rho h Gamma^2 by Newton's method."""
    d, e = u[0], u[4]
    m2 = (u[1:4] ** 2).sum(0)
    b2 = (b ** 2).sum(0)
    s = (u[1:4] * b).sum(0)
    k = (gam - 1) / gam
    a1, a0 = 4 / 3 * (b2 - e), (m2 + b2 * (b2 - 2 * e)) / 3      # v = 1: an upper bound
    W = 0.5 * (-a1 + torch.sqrt((a1 * a1 - 4 * a0).clamp(min=0)))
    W = torch.maximum(W, d) * (1 + 1e-9)

    def parts(W):
        v2 = (m2 * W * W + s * s * (2 * W + b2)) / _sq(W * (W + b2))
        v2 = v2.clamp(0, 1 - 1e-14)
        G = 1 / torch.sqrt(1 - v2)
        p = k * (W / (G * G) - d / G)
        return v2, G, p

    for _ in range(60):
        v2, G, p = parts(W)
        f = W - p + 0.5 * b2 * (1 + v2) - 0.5 * s * s / (W * W) - e
        dv = -2 / _sq(W) / W / (_sq(W + b2) * (W + b2)) * (
            s * s * (3 * W * (W + b2) + b2 * b2) + m2 * W * W * W)
        dp = k * (1 - v2 - W * dv + 0.5 * d * G * dv)
        df = 1 - dp + 0.5 * b2 * dv + s * s / (W * W * W)
        W = torch.maximum(W - f / df, 0.5 * W)
    v2, G, p = parts(W)
    v = (u[1:4] + (s / W) * b) / (W + b2)
    return torch.stack([d / G, G * v[0], G * v[1], G * v[2], p])


class _Grid:
    """Uniform global grid; arrays (..., k, j, i) of active cells or faces."""

    def __init__(self, m, dev):
        self.m, self.dev, self.g = m, dev, max(m.ng, 2)
        self.n = m.nx                                   # n1, n2, n3
        self.dx = [(m.xmax[d] - m.xmin[d]) / m.nx[d] for d in range(3)]
        self.gam = m.gamma
        self.floor = m.floors[0]
        self.solve = (_sr_hlle if m.relativistic else
                      (_hlld if m.rsolver == "hlld" else _hlle))

    def index(self, d, g, faces=False):
        n = self.n[d]
        i = torch.arange(-g, n + g + (1 if faces else 0), device=self.dev)
        if self.m.bc[2 * d] == "periodic":
            return torch.where((i == n) & faces, torch.full_like(i, n), i % n)
        return i.clamp(0, n if faces else n - 1)

    def pad(self, a, g, comp=-1):
        for d, axis in ((0, -1), (1, -2), (2, -3)):
            a = a.index_select(a.dim() + axis, self.index(d, g, d == comp))
        return a

    def centre(self, b):
        return torch.stack([0.5 * (b[0][:, :, 1:] + b[0][:, :, :-1]),
                            0.5 * (b[1][:, 1:] + b[1][:, :-1]), 0.5 * (b[2][1:] + b[2][:-1])])

    def primitives(self, u, b):
        c = self.centre(b)
        if self.m.relativistic:
            return _sr_primitives(u, c, self.gam), c
        d = u[0].clamp(min=self.floor)
        v = u[1:4] / d
        p = (self.gam - 1) * (u[4] - 0.5 * d * (v ** 2).sum(0) - 0.5 * (c ** 2).sum(0))
        return torch.stack([d, v[0], v[1], v[2], p.clamp(min=self.floor)]), c

    def conserved(self, w, c):
        if self.m.relativistic:
            x, y, z = w[1], w[2], w[3]
            u0 = torch.sqrt(1 + x * x + y * y + z * z)
            b0 = c[0] * x + c[1] * y + c[2] * z
            h = [(c[k] + b0 * w[k + 1]) / u0 for k in range(3)]
            bb = h[0] ** 2 + h[1] ** 2 + h[2] ** 2 - b0 * b0
            t = (w[0] + self.gam / (self.gam - 1) * w[4] + bb) * u0 * u0
            return torch.stack([w[0] * u0] + [t * w[k + 1] / u0 - b0 * h[k] for k in range(3)] +
                               [t - b0 * b0 - w[4] - 0.5 * bb])
        e = w[4] / (self.gam - 1) + 0.5 * w[0] * (w[1:4] ** 2).sum(0) + 0.5 * (c ** 2).sum(0)
        return torch.stack([w[0], w[0] * w[1], w[0] * w[2], w[0] * w[3], e])

    def fluxes(self, w, c, b, order, dt):
        """w, c padded by self.g, b the faces padded by 1: fluxes, face EMFs and upwind
        weights on the active faces and one transverse ghost layer."""
        g, out = self.g, []
        for d in range(3):
            t1, t2 = (d + 1) % 3, (d + 2) % 3
            q = torch.stack([w[0], w[1 + d], w[1 + t1], w[1 + t2], w[4], c[t1], c[t2]])
            # transverse: one ghost layer; the normal axis last
            sl = [slice(None)] * 4
            for t in (t1, t2):
                sl[3 - t] = slice(g - 1, g + self.n[t] + 1)
            q = q[tuple(sl)].movedim(3 - d, -1)
            fl = [slice(None)] * 3
            fl[2 - d] = slice(1, 1 + self.n[d] + 1)
            bn = b[d][tuple(fl)].movedim(2 - d, -1)
            L, R = _states(q, g, order)
            if order == 3:
                L, R = L.clone(), R.clone()
                for s in (L, R):
                    s[0].clamp_(min=self.floor)
                    s[4].clamp_(min=self.floor)
            f = self.solve(L, R, bn, self.gam)
            wt = 0.5 + (1024 * dt * f[0] / (self.dx[d] * (L[0] + R[0]))).clamp(-0.5, 0.5)
            f = f.movedim(-1, 3 - d)
            wt = wt.movedim(-1, 2 - d)
            flux = [None] * 5
            flux[0], flux[4] = f[0], f[4]
            flux[1 + d], flux[1 + t1], flux[1 + t2] = f[1], f[2], f[3]
            # E_{t2} = -F(B_t1), E_{t1} = F(B_t2)
            out.append((torch.stack(flux), {t2: -f[5], t1: f[6]}, wt))
        return out

    def corner(self, w, c, F):
        """Upwinded corner EMFs along each direction (Gardiner & Stone 2005), edge arrays of
        n + 1 positions across and n along."""
        v = w[1:4]
        if self.m.relativistic:
            v = v / torch.sqrt(1 + (v ** 2).sum(0))
        E = []
        for d in range(3):
            a, b = (d + 1) % 3, (d + 2) % 3
            g = self.g
            sl = tuple(slice(g - 1, g + self.n[x] + 1) if x != d else slice(g, g + self.n[x])
                       for x in (2, 1, 0))
            cc = (v[b] * c[a] - v[a] * c[b])[sl]              # along d, one ghost across

            def face(n, arr):                                 # faces normal to n, all of them
                s = tuple(slice(None) if x != d else slice(1, 1 + self.n[x])
                          for x in (2, 1, 0))
                return arr[s]

            Ea, Eb = face(a, F[a][1][d]), face(b, F[b][1][d])
            Wa, Wb = face(a, F[a][2]), face(b, F[b][2])

            def lo(x, axis):
                return x.narrow(2 - axis, 0, x.shape[2 - axis] - 1)

            def hi(x, axis):
                return x.narrow(2 - axis, 1, x.shape[2 - axis] - 1)

            # faces normal to a at low / high b, faces normal to b at low / high a
            Eal, Eah, Wal, Wah = lo(Ea, b), hi(Ea, b), lo(Wa, b), hi(Wa, b)
            Ebl, Ebh, Wbl, Wbh = lo(Eb, a), hi(Eb, a), lo(Wb, a), hi(Wb, a)
            ll, lh = lo(lo(cc, a), b), hi(lo(cc, a), b)       # (low a, low b), (low a, high b)
            hl, hh = lo(hi(cc, a), b), hi(hi(cc, a), b)
            # differences across, taken upwind by the mass flux
            dbl = (1 - Wal) * (Ebh - hl) + Wal * (Ebl - ll)
            dbh = (1 - Wah) * (Ebh - hh) + Wah * (Ebl - lh)
            dal = (1 - Wbl) * (Eah - lh) + Wbl * (Eal - ll)
            dah = (1 - Wbh) * (Eah - hh) + Wbh * (Eal - hl)
            E.append(0.25 * (dbl + dbh + dal + dah + Eal + Eah + Ebl + Ebh))
        return E

    def divergence(self, F):
        out = 0
        for d in range(3):
            f = F[d][0]
            for t in ((d + 1) % 3, (d + 2) % 3):
                f = f.narrow(3 - t, 1, self.n[t])
            out = out + (f.narrow(3 - d, 1, self.n[d]) - f.narrow(3 - d, 0, self.n[d])) / self.dx[d]
        return out

    def curl(self, E):
        out = []
        for d in range(3):
            a, b = (d + 1) % 3, (d + 2) % 3
            da = lambda x: (x.narrow(2 - a, 1, self.n[a]) - x.narrow(2 - a, 0, self.n[a])) / self.dx[a]  # noqa: E731,B023
            db = lambda x: (x.narrow(2 - b, 1, self.n[b]) - x.narrow(2 - b, 0, self.n[b])) / self.dx[b]  # noqa: E731,B023
            out.append(da(E[b]) - db(E[a]))
        return out

    def step(self, w, c, b, u0, b0, order, dt, dtw):
        wp, cp = self.pad(w, self.g), self.centre([self.pad(b[q], self.g, q) for q in range(3)])
        bp = [self.pad(b[q], 1, q) for q in range(3)]
        F = self.fluxes(wp, cp, bp, order, dtw)
        E = self.corner(wp, cp, F)
        return (u0 - dt * self.divergence(F),
                [x - dt * y for x, y in zip(b0, self.curl(E))])

    def new_dt(self, w, c, b):
        m, out = self.m, math.inf
        for d in range(3):
            s = torch.ones_like(w[0])
            if not m.relativistic:
                t1, t2 = (d + 1) % 3, (d + 2) % 3
                lowf = b[d].narrow(2 - d, 0, self.n[d])
                q = torch.stack([w[0], w[1 + d], w[1 + t1], w[1 + t2], w[4], c[t1], c[t2]])
                s = w[1 + d].abs() + _fast(q, c[d] + (lowf - c[d]).abs(), self.gam)
            out = min(out, float((self.dx[d] / s).min()))
        return out * m.cfl

    def run(self, u, b, cycles):
        w, c = self.primitives(u, b)
        t, dt = 0.0, self.new_dt(w, c, b)
        for _ in range(cycles):
            uh, bh = self.step(w, c, b, u, b, 1, 0.5 * dt, dt)
            wh, ch = self.primitives(uh, bh)
            u, b = self.step(wh, ch, bh, u, b, self.m.xorder, dt, dt)
            w, c = self.primitives(u, b)
            t, dt = t + dt, min(2 * dt, self.new_dt(w, c, b))
        return u, b, w, t, dt

    def blocks(self, u, b, w):
        """The registers of every MeshBlock, ghosts included, stacked."""
        m, g = self.m, self.m.ng
        n1, n2, n3 = m.bnx
        bp = [self.pad(b[q], g, q) for q in range(3)]
        # across an open face the ghost state is rebuilt from the copied primitives
        up = self.conserved(self.pad(w, g), self.centre(bp)) if "outflow" in m.bc else self.pad(u, g)
        if "outflow" in m.bc:
            up[:, g:-g, g:-g, g:-g] = u
        out = {k: [] for k in KEYS}
        for gid in range(m.nblocks):
            l1, l2, l3 = m.loc(gid)
            k, j, i = l3 * n3, l2 * n2, l1 * n1
            e3, e2, e1 = k + n3 + 2 * g, j + n2 + 2 * g, i + n1 + 2 * g
            out["u"].append(up[:, k:e3, j:e2, i:e1])
            out["b1"].append(bp[0][k:e3, j:e2, i:e1 + 1])
            out["b2"].append(bp[1][k:e3, j:e2 + 1, i:e1])
            out["b3"].append(bp[2][k:e3 + 1, j:e2, i:e1])
        return {k: torch.stack(v) for k, v in out.items()}


def _gather(m, problem, dev):
    """Active conserved state of the global grid from the problem generator's MeshBlocks."""
    n1, n2, n3 = m.nx
    g = m.ng
    u = np.zeros((5, n3, n2, n1))
    b = [np.zeros((n3, n2, n1 + 1)), np.zeros((n3, n2 + 1, n1)), np.zeros((n3 + 1, n2, n1))]
    c1, c2, c3 = m.bnx
    for gid in range(m.nblocks):
        l1, l2, l3 = m.loc(gid)
        a = problem.block(gid)
        K, J, I = l3 * c3, l2 * c2, l1 * c1
        u[:, K:K + c3, J:J + c2, I:I + c1] = a["u"][:, g:g + c3, g:g + c2, g:g + c1]
        b[0][K:K + c3, J:J + c2, I:I + c1 + 1] = a["b1"][g:g + c3, g:g + c2, g:g + c1 + 1]
        b[1][K:K + c3, J:J + c2 + 1, I:I + c1] = a["b2"][g:g + c3, g:g + c2 + 1, g:g + c1]
        b[2][K:K + c3 + 1, J:J + c2, I:I + c1] = a["b3"][g:g + c3 + 1, g:g + c2, g:g + c1]
    to = lambda x: torch.from_numpy(x).to(dev)  # noqa: E731
    return to(u), [to(x) for x in b]


def _exact_mesh(m, problem, cycles, dev):
    grid = _Grid(m, dev)
    u, b = _gather(m, problem, dev)
    u, b, w, t, dt = grid.run(u, b, cycles)
    return grid.blocks(u, b, w), [t, dt, cycles]


def exact(case, seed):
    dev = torch.device("cuda:0" if torch.cuda.is_available() else "cpu")
    kind = case["kind"]
    if kind == "refined":
        return None        # a second multilevel code would be needed
    if kind == "recover":
        cons, bcc, _ = ml.conserved_batch(case["n"], seed)
        w = _sr_primitives(torch.from_numpy(cons).to(dev).T, torch.from_numpy(bcc).to(dev).T,
                           ml.GAMMA_AD)
        return {"cons": torch.from_numpy(cons), "prim": w.T.contiguous()}
    if kind == "block":
        return _exact_block(case, seed, dev)
    if float(_cells(case)) * case["cycles"] > 2.5e8:
        return None        # more than about 20 s in plain torch
    if kind == "ensemble":
        return [_exact_mesh(m, p, case["cycles"], dev)[0]
                for m, p in _ensemble_members(case, seed)]
    m = _mesh(case)
    if m.relativistic and m.rsolver == "hlld":
        return None        # its iteration on the contact pressure has no closed form
    out, clock = _exact_mesh(m, _problem(case, m, seed), case["cycles"], dev)
    return dict(out, clock=clock)


def _exact_block(case, seed, dev):
    m, dt, (w, bcc, u0), f = _block_state(case, seed, dev)
    grid = _Grid(m, dev)
    g = m.ng
    n = m.nx
    cut = []
    for q in range(3):
        s = [slice(g - 1, -(g - 1)) if g > 1 else slice(None)] * 3
        cut.append(f[q][tuple(s)])
    F = grid.fluxes(w, bcc, cut, case["order"], dt)
    E = grid.corner(w, bcc, F)
    act = (slice(g, -g),) * 3
    u = u0.clone()
    u[(slice(None),) + act] -= dt * grid.divergence(F)
    b = [x.clone() for x in f]
    for q, y in enumerate(grid.curl(E)):
        s = [slice(g, -g)] * 3
        b[q][tuple(s)] -= dt * y
    wo, co = grid.primitives(u, b)
    inner = grid.primitives(u[(slice(None),) + act], [x[act] for x in b])
    ndt = grid.new_dt(inner[0], inner[1], [x[act] for x in b])
    e, flux = [], []
    for d in range(3):
        c1, c2, c3 = m.nc
        fs = [(c3, c2, c1 + 1), (c3, c2 + 1, c1), (c3 + 1, c2, c1)][d]
        e.append(None)     # the library fills one more layer of edge positions
        y = torch.zeros((5,) + fs, dtype=torch.float64, device=dev)
        s = [slice(g - 1, g + n[x] + 1) if x != d else slice(g, g + n[d] + 1)
             for x in (2, 1, 0)]
        y[(slice(None),) + tuple(s)] = F[d][0]
        flux.append(y)
    return {"u": u, "b": b, "w": wo, "bcc": co,
            "dt": torch.tensor([ndt], dtype=torch.float64, device=dev), "e": e, "flux": flux}
