"""Workloads of the framework's solvers, for timing and for comparing results.

Every case is one stretch of work a user's program has the framework do
between two looks at the results: so many time steps of a resident solve and
the read-back of its fields, a batch or a union of solves, an implicit
advection-diffusion stage, a free-form deformation.  Sizes follow bench.py's
workloads (the 20^3 cavity, the 96^3 channel, the 128^3 hexa cavity, the
serving and batch mixes) and odd sizes between and below them.

    listed()            the cases, each a dict of plain values
    draw(rng)           one more case of the same ranges
    prepare(case, seed) mesh, boundary conditions, handles and initial state
    run(state)          one pass through the public entry points
    work(case)          bytes and flops one pass cannot do without
    exact(case, seed)   the first pass's results in plain 64-bit torch
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from femorph_amd import femx, meshgen
from femorph_amd.mesh import Mesh

PRECISION = {"fp64": femx.FEMX_FP64, "mixed": femx.FEMX_MIXED}
REYNOLDS = {"vms": 200.0, "supg": 400.0}


def listed():
    return [
        # the smallest everyday solve: 48k tets, where launches and latency count
        dict(name="vms cavity 20 mixed", kind="vms", flow="cavity", nx=20, ny=20, nz=20, precision="mixed", dual=0,
             norms=0, steps=100),
        # the headline solve: 5.3M tets, inflow, walls and a pressure outlet
        dict(name="vms channel 96 mixed", kind="vms", flow="channel", nx=96, ny=96, nz=96, precision="mixed", dual=0,
             norms=0, steps=200),
        # the default precision of the drop-in classes, a box of unequal odd sides
        dict(name="vms channel 71x53x61 fp64", kind="vms", flow="channel", nx=71, ny=53, nz=61, precision="fp64",
             dual=0, norms=0, steps=60),
        # what the drop-in solve runs: dual iterations and the printed per-iteration norms
        dict(name="vms cavity 33 dual norms fp64", kind="vms", flow="cavity", nx=33, ny=33, nz=33, precision="fp64",
             dual=1, norms=1, steps=30),
        # many small cavities advanced together, each its own Reynolds number
        dict(name="vms batch 32 mixed", kind="batch", members=32, n_min=8, n_max=40, precision="mixed", steps=50),
        # resident solves of mixed sizes joined for a stretch of steps, as the solve server does
        dict(name="vms union 10", kind="union", solver="vms", members=10, n_min=8, n_max=48, steps=40),
        dict(name="supg union 10", kind="union", solver="supg", members=10, n_min=8, n_max=40, steps=40),
        # 2.1M hexahedra, lid-driven, between two saves
        dict(name="supg cavity 128 mixed", kind="supg", elem="hexa8", nx=128, ny=128, nz=128, precision="mixed",
             steps=100),
        # the drop-in classes' default precision on hexahedra, odd sides
        dict(name="supg cavity 45x37x51 fp64", kind="supg", elem="hexa8", nx=45, ny=37, nz=51, precision="fp64",
             steps=50),
        # a small tetrahedral SUPG solve
        dict(name="supg cavity 17 tet4 fp64", kind="supg", elem="tet4", nx=17, ny=17, nz=17, precision="fp64",
             steps=50),
        # implicit advection-diffusion: assembly, GMRES to 1e-5, update, a few time steps
        dict(name="advdiff 57 tet4", kind="ins", elem="tet4", nx=57, ny=57, nz=57, steps=4),
        # a morph of half a million resident mesh nodes by a moderate control lattice
        dict(name="ffd 500k 7x6x5", kind="ffd", points=500_009, lx=7, ly=6, lz=5, displaced=24),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _sides(rng, lo, hi):
    """Three sides around one log-uniform size, each varied by a fifth."""
    n = _log_int(rng, lo, hi)
    return [max(3, min(hi, int(round(n * rng.uniform(0.8, 1.25))))) for _ in range(3)]


def draw(rng):
    kind = rng.choice(["vms", "vms", "vms", "supg", "supg", "supg", "batch", "union", "ins", "ffd"])
    if kind == "vms":
        nx, ny, nz = _sides(rng, 8, 72)
        precision = rng.choice(["mixed", "fp64"])
        return dict(kind="vms", flow=rng.choice(["cavity", "channel"]), nx=nx, ny=ny, nz=nz, precision=precision,
                    dual=rng.choice([0, 0, 0, 1]),
                    norms=rng.choice([0, 0, 1]) if precision == "fp64" and nx * ny * nz < 64000 else 0,
                    steps=rng.randrange(20, 101))
    if kind == "supg":
        elem = rng.choice(["hexa8", "hexa8", "tet4"])
        nx, ny, nz = _sides(rng, 6, 96 if elem == "hexa8" else 40)
        return dict(kind="supg", elem=elem, nx=nx, ny=ny, nz=nz, precision=rng.choice(["mixed", "fp64"]),
                    steps=rng.randrange(20, 101))
    if kind == "batch":
        return dict(kind="batch", members=rng.randrange(4, 41), n_min=rng.randrange(4, 12),
                    n_max=rng.randrange(16, 37), precision=rng.choice(["mixed", "mixed", "fp64"]),
                    steps=rng.randrange(10, 61))
    if kind == "union":
        return dict(kind="union", solver=rng.choice(["vms", "supg"]), members=rng.randrange(2, 13),
                    n_min=rng.randrange(6, 12), n_max=rng.randrange(16, 41), steps=rng.randrange(10, 61))
    if kind == "ins":
        elem = rng.choice(["tet4", "tet4", "hexa8"])
        nx, ny, nz = _sides(rng, 8, 64 if elem == "tet4" else 48)
        return dict(kind="ins", elem=elem, nx=nx, ny=ny, nz=nz, steps=rng.randrange(2, 6))
    lx, ly, lz = (rng.randrange(2, 14) for _ in range(3))
    return dict(kind="ffd", points=_log_int(rng, 1_000, 600_000), lx=lx, ly=ly, lz=lz, displaced=rng.randrange(1, 65))


# ------------------------------------------------------------------ inputs

_TETS = [[v[0] + 2 * v[1] + 4 * v[2] for v in verts] for verts in meshgen._KUHN]
_HEXA = [v[0] + 2 * v[1] + 4 * v[2] for v in meshgen._HEX_LOCAL]


def _box(nx, ny, nz, elem, jitter, rng):
    """The unit cube cut into nx * ny * nz boxes, each six tets or one hexa,
    interior node components jittered by a fraction of the spacing."""
    axes = [np.linspace(0.0, 1.0, n + 1) for n in (nx, ny, nz)]
    xyz = np.empty((nz + 1, ny + 1, nx + 1, 3))
    xyz[..., 0], xyz[..., 1], xyz[..., 2] = axes[0], axes[1][:, None], axes[2][:, None, None]
    for c, (n, ax) in enumerate(((nx, 2), (ny, 1), (nz, 0))):
        inner = [slice(None)] * 3
        inner[ax] = slice(1, -1)
        part = xyz[tuple(inner) + (c,)]
        part += (jitter / n) * (2.0 * rng.random(part.shape) - 1.0)
    corner = [i + (nx + 1) * (j + (ny + 1) * k) for k in (0, 1) for j in (0, 1) for i in (0, 1)]
    i, j, k = (np.arange(n, dtype=np.int32) for n in (nx, ny, nz))
    first = (i + (nx + 1) * (j[:, None] + (ny + 1) * k[:, None, None])).astype(np.int32).reshape(-1, 1)
    local = np.array(_TETS if elem == "tet4" else [_HEXA])
    conn = first + np.array(corner, np.int32)[local].reshape(1, -1)
    return Mesh(xyz.reshape(-1, 3), conn.reshape(-1, local.shape[1]))


def _tet_h(mesh):
    x = mesh.coords[mesh.conn[::max(1, mesh.n_elems // 200_000)]]
    return float(np.cbrt(np.abs(np.linalg.det(x[:, 1:] - x[:, :1])).min()))


def _vms_parts(nx, ny, nz, flow, rng, re=None, dual=0):
    mesh = _box(nx, ny, nz, "tet4", 0.15, rng)
    bc = meshgen.channel_bc(mesh) if flow == "channel" else meshgen.lid_cavity_bc(mesh)
    prm = dict(rho=1.0, mu=1.0 / (re or REYNOLDS["vms"]), inv_eps=1.0, c1=4.0, c2=2.0, dt=0.1 * _tet_h(mesh),
               tot_dual_steps=dual)
    return mesh, bc, prm, _start(mesh, rng, 4)


def _supg_parts(nx, ny, nz, elem, rng, re=None):
    mesh = _box(nx, ny, nz, elem, 0.2 if elem == "hexa8" else 0.15, rng)
    prm = dict(rho=1.0, mu=1.0 / (re or REYNOLDS["supg"]), alpha=1.0, cI=4.0, dt=0.1 / max(nx, ny, nz))
    if elem == "tet4":
        prm["exopts"] = (0, 0, 1, 1, 1, 1)  # B-hat needs hexahedra
    return mesh, meshgen.lid_cavity_bc(mesh), prm, _start(mesh, rng, 3)


def _start(mesh, rng, dofs):
    """A smooth swirl with a little noise, as a flow under way has."""
    x, y, z = mesh.coords.T
    a, b, c = rng.uniform(0.1, 0.3, 3)
    u = np.zeros((mesh.n_nodes, dofs))
    u[:, 0] = a * np.sin(math.pi * x) * np.cos(math.pi * y)
    u[:, 1] = -b * np.cos(math.pi * x) * np.sin(math.pi * y)
    u[:, 2] = c * np.sin(2 * math.pi * z) * np.sin(math.pi * x)
    u[:, :3] += 1e-3 * (2.0 * rng.random((mesh.n_nodes, 3)) - 1.0)
    return u


def _member_sizes(case):
    """Log-uniform sizes spread evenly over the range, the largest included."""
    at = (np.arange(case["members"]) + 0.5) / case["members"]
    lo, hi = math.log(case["n_min"]), math.log(case["n_max"])
    return [int(round(math.exp(lo + t * (hi - lo)))) for t in at[:-1]] + [case["n_max"]]


def _batch_parts(case, rng):
    return [_vms_parts(n, n, n, "cavity", rng, re=rng.uniform(50.0, 500.0)) for n in _member_sizes(case)]


def _union_parts(case, rng):
    if case["solver"] == "vms":
        return [_vms_parts(n, n, n, "cavity", rng) for n in _member_sizes(case)]
    return [_supg_parts(n, n, n, "hexa8", rng, re=200.0) for n in _member_sizes(case)]


def _ins_parts(case, rng):
    mesh = _box(case["nx"], case["ny"], case["nz"], case["elem"], 0.15, rng)
    c = mesh.coords
    wall = np.nonzero((c.min(axis=1) < 1e-12) | (c.max(axis=1) > 1 - 1e-12))[0].astype(np.int32)
    mid = rng.uniform(0.35, 0.65, 3)
    phi = np.exp(-40.0 * ((c - mid) ** 2).sum(axis=1))
    phi[wall] = 0.0
    am, af = 0.5 * 2.5 / 1.5, 1.0 / 1.5  # generalized-alpha, rho_inf = 0.5
    prm = dict(dt=0.5 / max(case["nx"], case["ny"], case["nz"]), alpha_m=am, alpha_f=af, gamma=0.5 + am - af)
    diff = rng.uniform(0.2e-3, 1.0e-3, (mesh.n_elems, 3))
    return mesh, wall, phi, diff, prm


def _ffd_parts(case, rng):
    n = (case["lx"], case["ly"], case["lz"])
    tot = n[0] * n[1] * n[2]
    nodes = rng.choice(tot, min(case["displaced"], tot), replace=False).astype(np.int32)
    box = ((0.05, -0.1, 0.02), n, (0.9, 0.1, 0.0), (0.05, 1.1, 0.1), (0.0, -0.1, 0.9))
    return box, nodes, rng.uniform(-0.2, 0.2, (len(nodes), 3)), rng.random((case["points"], 3))


# ----------------------------------------------------------------- passes

def _ptr(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))


def _vms_solver(mesh, bc, prm, start, precision):
    s = femx.VMSSolver(femx.DeviceMesh(mesh), bc, precision=PRECISION[precision], **prm)
    s.set_state(start)
    return s


def _supg_solver(mesh, bc, prm, start, precision):
    s = femx.SUPGSolver(femx.DeviceMesh(mesh), bc, precision=PRECISION[precision], **prm)
    s.set_state(start)
    return s


def _vms_fields(mesh):
    return dict(sol=np.zeros((mesh.n_nodes, 4)))


def _supg_fields(mesh):
    return dict(sol=np.zeros((mesh.n_nodes, 3)), pres=np.zeros(mesh.n_elems), lam=np.zeros(mesh.n_elems))


def _vms_read(s, f):
    """Velocity and pressure of every node (femx_vms_get_state; the subgrid
    velocities stay on the device, as between two saves)."""
    femx._check(femx.load().femx_vms_get_state(s._h, _ptr(f["sol"]), None, None))
    return f


def _supg_read(s, f):
    """Velocity, element pressure and element bulk modulus (femx_supg_get_state)."""
    femx._check(femx.load().femx_supg_get_state(s._h, _ptr(f["sol"]), _ptr(f["pres"]), _ptr(f["lam"]), None, None))
    return f


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind, st = case["kind"], dict(case=case)
    if kind == "vms":
        mesh, bc, prm, start = _vms_parts(case["nx"], case["ny"], case["nz"], case["flow"], rng, dual=case["dual"])
        st["solver"] = _vms_solver(mesh, bc, prm, start, case["precision"])
        st["fields"] = _vms_fields(mesh)
        if case["norms"]:
            st["solver"].set_diagnostics(2)
    elif kind == "supg":
        mesh, bc, prm, start = _supg_parts(case["nx"], case["ny"], case["nz"], case["elem"], rng)
        st["solver"] = _supg_solver(mesh, bc, prm, start, case["precision"])
        st["fields"] = _supg_fields(mesh)
    elif kind == "batch":
        parts = _batch_parts(case, rng)
        st["batch"] = femx.VMSBatch([(m, bc, dict(p, precision=PRECISION[case["precision"]])) for m, bc, p, _ in parts])
        st["batch"].set_state([s for _, _, _, s in parts])
    elif kind == "union":
        parts = _union_parts(case, rng)
        vms = case["solver"] == "vms"
        st["union"] = femx.VMSUnion() if vms else femx.SUPGUnion()
        st["solvers"] = [(_vms_solver if vms else _supg_solver)(*p, "mixed") for p in parts]
        st["fields"] = [(_vms_fields if vms else _supg_fields)(p[0]) for p in parts]
    elif kind == "ins":
        mesh, wall, phi, diff, prm = _ins_parts(case, rng)
        st["solver"] = femx.INSSolver(femx.DeviceMesh(mesh), el_diff=diff, dir_node=wall,
                                      dir_val=np.zeros((len(wall), 3)), **prm)
        st["solver"].set_state(phi=phi, phi_dot=np.zeros(mesh.n_nodes))
        st.update(time=0.0, dt=prm["dt"])
    else:
        box, nodes, vals, points = _ffd_parts(case, rng)
        st.update(box=box, nodes=nodes, vals=vals, points=torch.from_numpy(points).cuda())
        st["moved"] = torch.zeros_like(st["points"])
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "vms":
        s = st["solver"]
        s.step(case["steps"])
        out = _vms_read(s, st["fields"])
        return dict(out, norms=s.get_norms(min(case["steps"], 64))) if case["norms"] else out
    if kind == "supg":
        st["solver"].step(case["steps"])
        return _supg_read(st["solver"], st["fields"])
    if kind == "batch":
        st["batch"].step(case["steps"])
        return [st["batch"].get_state(i)[0] for i in range(case["members"])]
    if kind == "union":
        # members run their first step alone, then join
        u, vms = st["union"], case["solver"] == "vms"
        for s in st["solvers"]:
            s.step(1) if vms else s.step_async(1)
            u.add(s, case["steps"] - 1)
        u.step(case["steps"] - 1)
        for s in st["solvers"]:
            u.remove(s)
        if not vms:
            for s in st["solvers"]:
                s.finish()
        return [(_vms_read if vms else _supg_read)(s, f) for s, f in zip(st["solvers"], st["fields"])]
    if kind == "ins":
        s = st["solver"]
        for _ in range(case["steps"]):
            s.prescribe_velocity(0, st["time"])
            s.advdiff_solve()
            s.update()
            st["time"] += st["dt"]
        phi, phi_dot, vel = s.get_state()
        return dict(phi=phi, phi_dot=phi_dot, vel=vel)
    femx.ffd_morph_noalloc(*st["box"], st["nodes"], st["vals"], case["points"], st["points"].data_ptr(),
                           st["moved"].data_ptr(), torch.cuda.current_stream().cuda_stream)
    return st["moved"]


# ------------------------------------------------------------------- work

def _mean_cube(case):
    lo, hi = case["n_min"], case["n_max"]
    return (hi ** 3 - lo ** 3) / (3.0 * math.log(hi / lo)) if hi > lo else hi ** 3


def _vms_work(boxes, steps, precision, dual):
    e, n, wide = 6.0 * boxes, float(boxes), 8 if precision == "fp64" else 4
    # connectivity, subgrid velocities read and written; per node coordinates, mass, state read and written
    step = e * (16 + 24 * wide) + n * (3 * wide + 8 + 64)
    return dict(bytes=steps * (dual + 1) * step + 32 * n, flops=steps * (dual + 1) * e * 1000.0)


def _supg_work(boxes, steps, elem):
    e, n, npe = boxes * (6.0 if elem == "tet4" else 1.0), float(boxes), 4 if elem == "tet4" else 8
    # connectivity, bulk modulus; per node coordinates, mass, velocity and nodal force read and written
    step = e * (4 * npe + 8) + n * (32 + 48 + 48)
    return dict(bytes=steps * step + 24 * n + 16 * e, flops=steps * e * (900.0 if elem == "tet4" else 5500.0))


def work(case):
    kind = case["kind"]
    if kind in ("vms", "supg", "ins"):
        boxes = case["nx"] * case["ny"] * case["nz"]
    if kind == "vms":
        return _vms_work(boxes, case["steps"], case["precision"], case["dual"])
    if kind == "supg":
        return _supg_work(boxes, case["steps"], case["elem"])
    if kind == "batch":
        return _vms_work(case["members"] * _mean_cube(case), case["steps"], case["precision"], 0)
    if kind == "union":
        boxes = case["members"] * _mean_cube(case)
        return (_vms_work(boxes, case["steps"], "mixed", 0) if case["solver"] == "vms"
                else _supg_work(boxes, case["steps"], "hexa8"))
    if kind == "ins":
        tet = case["elem"] == "tet4"
        e, n, nnz, its = boxes * (6.0 if tet else 1.0), float(boxes), boxes * (15.0 if tet else 27.0), 8
        # assembly; per Krylov iteration the matrix, the vector and the basis once
        step = e * (24 if tet else 40) + n * 72 + nnz * 8 + its * (nnz * 12 + n * 8 * (3 + its / 2.0))
        return dict(bytes=case["steps"] * step, flops=case["steps"] * (e * (600.0 if tet else 6000.0) + its * nnz * 2))
    cells = case["lx"] * case["ly"] * case["lz"]
    return dict(bytes=48.0 * case["points"], flops=case["points"] * 6.0 * cells)


# ------------------------------------------------------------- exact values
# The same methods written plainly with torch in 64 bits.

def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _t(a, dtype=torch.float64):
    return torch.as_tensor(np.ascontiguousarray(a), device=_dev()).to(dtype)


def _node_sum(conn, values, n):
    """Sum of element-corner values [E, npe, k] at the nodes."""
    out = torch.zeros((n, values.shape[-1]), dtype=torch.float64, device=values.device)
    return out.index_add_(0, conn.reshape(-1), values.reshape(-1, values.shape[-1]))


class _Conditions:
    """Constant velocity tables, then pressures, then fixed walls."""

    def __init__(self, bc):
        first = np.asarray(bc.vel_row_off[:-1])
        self.vel, self.vel_at = _t(bc.vel_node, torch.long), _t(bc.vel_rows[first][:, :3])
        self.wall, self.wall_at = _t(bc.dir_node, torch.long), _t(bc.dir_val)
        self.pres, self.pres_at = _t(bc.pres_node, torch.long), _t(bc.pres_val)

    def __call__(self, sol):
        sol = sol.clone()
        sol[self.vel, :3] = self.vel_at
        if sol.shape[1] > 3:
            sol[self.pres, 3] = self.pres_at
        sol[self.wall, :3] = self.wall_at
        return sol


def _vms_exact(parts, steps):
    mesh, bc, prm, start = parts
    n, conn, fix = mesh.n_nodes, _t(mesh.conn, torch.long), _Conditions(bc)
    x = _t(mesh.coords)[conn]
    edge = (x[:, 1:] - x[:, :1]).transpose(1, 2)
    inv, six_v = _inv3(edge), _det3(edge)
    grad = torch.cat([-inv.sum(1, keepdim=True), inv], 1)  # [E, 4, 3]
    vol, h = six_v / 6.0, six_v.pow(1.0 / 3.0)
    mass = _node_sum(conn, (vol / 4.0)[:, None, None].expand(-1, 4, 1), n)
    ga, gb = 0.58541020, 0.13819660
    shape = torch.full((4, 4), gb, dtype=torch.float64, device=x.device).fill_diagonal_(ga)
    nu, dt, w = prm["mu"] / prm["rho"], prm["dt"], (vol / 4.0)[:, None]
    q = fix(_t(start))
    p, sub, said = q, torch.zeros((4, mesh.n_elems, 3), dtype=torch.float64, device=x.device), []
    pending = False

    def times(g, v):  # (v . grad) u for g = du_i / dx_j
        return (g * v[:, None, :]).sum(-1)

    for _ in range(steps):
        for d in range(prm["tot_dual_steps"] + 1):
            if pending:  # projection of the residual and the subgrid velocities of the iteration before
                u = p[:, :3][conn]
                g = (u[:, :, :, None] * grad[:, :, None, :]).sum(1)
                dp = (grad * p[:4, 3][None, :, None]).sum(1)
                conv = [(shape[k][None, :, None] * u).sum(1) + sub[k] for k in range(4)]
                res = [times(g, c) + dp for c in conv]
                speed = torch.stack([(c * c).sum(1) for c in conv]).amax(0).sqrt()
                tau = 1.0 / (1.0 / dt + prm["c1"] * nu / h ** 2 + prm["c2"] * speed / h)
                nodal = [sum(shape[k][b] * res[k] for k in range(4)) / (ga + 3 * gb) for b in range(4)]
                sub = torch.stack([(sub[k] / dt - res[k] + sum(shape[k][b] * nodal[b] for b in range(4)))
                                   * tau[:, None] for k in range(4)])
            u, pe = q[:, :3][conn], q[:, 3][conn]
            g = (u[:, :, :, None] * grad[:, :, None, :]).sum(1)
            div = g.diagonal(dim1=1, dim2=2).sum(1)[:, None]
            old = (u - p[:, :3][conn]) / dt if d > 0 else None
            r = torch.zeros((mesh.n_elems, 4, 4), dtype=torch.float64, device=x.device)
            for k in range(4):
                a = (shape[k][None, :, None] * u).sum(1) + sub[k]
                along = times(g, a)
                if d > 0:
                    along = along + (shape[k][None, :, None] * old).sum(1)
                pk = (shape[k][None, :] * pe).sum(1, keepdim=True)
                for b in range(4):
                    r[:, b, :3] += w * (shape[k][b] * along + nu * times(g, grad[:, b]) - pk * grad[:, b]
                                        - (grad[:, b] * a).sum(1, keepdim=True) * sub[k])
                    r[:, b, 3:] += w * prm["inv_eps"] * (shape[k][b] * div
                                                         - (grad[:, b] * sub[k]).sum(1, keepdim=True))
            p = (q if d == 0 else p) - dt / mass * _node_sum(conn, r, n)
            q = fix(p)
            pending = True
    return dict(sol=q)


def _det3(m):
    return (m[:, 0] * torch.linalg.cross(m[:, 1], m[:, 2])).sum(-1)


def _inv3(m):
    a, b, c = m[:, 0], m[:, 1], m[:, 2]
    rows = [torch.linalg.cross(b, c), torch.linalg.cross(c, a), torch.linalg.cross(a, b)]
    return torch.stack(rows, -1) / _det3(m)[:, None, None]


def _shapes(npe):
    """Values and local derivatives at the second-order Gauss points, and the weight."""
    if npe == 4:
        ga, gb = 0.58541020, 0.13819660
        pts = np.array([[ga, gb, gb], [gb, ga, gb], [gb, gb, ga], [gb, gb, gb]])
        val = np.concatenate([pts, 1.0 - pts.sum(1, keepdims=True)], 1)
        return val, np.tile(np.vstack([np.eye(3), -np.ones((1, 3))]), (4, 1, 1)), 1.0 / 24.0
    s = np.array([[2 * i - 1 for i in v] for v in meshgen._HEX_LOCAL], float)
    f = 1.0 + s[:, None, :] * s[None, :, :] / math.sqrt(3.0)  # [point, node, axis]
    der = np.stack([s[None, :, 0] * f[..., 1] * f[..., 2], s[None, :, 1] * f[..., 0] * f[..., 2],
                    s[None, :, 2] * f[..., 0] * f[..., 1]], -1) / 8.0
    return f.prod(-1) / 8.0, der, 1.0


def _geometry(mesh):
    """Per Gauss point: inverse Jacobian [E, 3, 3], d N / d x [E, npe, 3] and det J * weight [E]."""
    conn = _t(mesh.conn, torch.long)
    x = _t(mesh.coords)[conn]
    x = x - x[:, :1]
    val, der, weight = _shapes(mesh.npe)
    points = []
    for g in range(len(val)):
        d = _t(der[g])
        jac = (d[None, :, :, None] * x[:, :, None, :]).sum(1)
        inv = _inv3(jac)
        points.append((inv, (inv[:, None] * d[None, :, None, :]).sum(-1), _det3(jac) * weight))
    return conn, _t(val), points


def _supg_exact(parts, steps):
    mesh, bc, prm, start = parts
    n, fix = mesh.n_nodes, _Conditions(bc)
    conn, val, points = _geometry(mesh)
    rho, mu, dt = prm["rho"], prm["mu"], prm["dt"]
    nu, bhat = mu / rho, "exopts" not in prm
    mass = _node_sum(conn, sum(rho * dv[:, None] * val[g][None, :] for g, (_, _, dv) in enumerate(points))[..., None], n)
    vol = sum(dv for _, _, dv in points)
    avg = sum(dn * dv[:, None, None] for _, dn, dv in points) / vol[:, None, None]
    metric = [(inv[:, :, :, None] * inv[:, :, None, :]).sum(1) for inv, _, _ in points]
    inverse = [_inv3(m) for m in metric]
    eye = torch.eye(3, dtype=torch.float64, device=val.device)
    sol, before = fix(_t(start)), None
    lam = None
    for _ in range(steps):
        u = sol[conn]
        out, lam, alpha = torch.zeros_like(u), 0.0, 0.0
        mean = (avg * u).sum(1) if bhat else None  # [E, 3]
        for g, (inv, dn, dv) in enumerate(points):
            ug = (val[g][None, :, None] * u).sum(1)
            gu = (dn[:, :, :, None] * u[:, :, None, :]).sum(1)  # du_i / dx_b
            div = gu.diagonal(dim1=1, dim2=2).sum(1)
            m = metric[g]
            tau = ((ug[:, :, None] * m * ug[:, None, :]).sum((1, 2)) + prm["cI"] * nu ** 2 * (m * m).sum((1, 2))).rsqrt()
            nu_c = 1.0 / (m.diagonal(dim1=1, dim2=2).sum(1) * tau)
            bulk = prm["alpha"] * (ug[:, :, None] * inverse[g] * ug[:, None, :]).sum((1, 2)).sqrt().clamp(min=nu)
            lam = lam + bulk * dv
            c = (ug[:, :, None] * gu).sum(1)
            eps = gu.diagonal(dim1=1, dim2=2)
            if bhat:
                b = (mean - eps) / 3.0
                eps = eps - 2.0 * b + b.sum(1, keepdim=True)
            s = 2.0 * mu * eps + (bulk * eps.sum(1))[:, None]
            if bhat:
                alpha = alpha + dv[:, None] * (s.sum(1, keepdim=True) - 2.0 * s) / 3.0
                s = (5.0 * s - s.sum(1, keepdim=True)) / 3.0
            shear = mu * (gu + gu.transpose(1, 2)) * (1.0 - eye)
            stress = (shear + torch.diag_embed(s) + (rho * nu_c * div)[:, None, None] * eye) * dv[:, None, None]
            along = rho * dv[:, None] * (val[g][None, :] + tau[:, None] * (dn * ug[:, None, :]).sum(-1))
            out += along[:, :, None] * c[:, None, :] + (dn[:, :, :, None] * stress[:, None]).sum(2)
        if bhat:
            out += avg * alpha[:, None, :]
        force = _node_sum(conn, -dt * out, n)
        sol = fix(sol + (force if before is None else 1.5 * force - 0.5 * before) / mass)
        before, lam = force, lam / vol
    u = sol[conn]
    div = sum((dn * u).sum((1, 2)) * dv for _, dn, dv in points) / vol
    return dict(sol=sol, pres=-lam * div, lam=lam)


def _ins_exact(case, rng):
    mesh, wall, phi, diff, prm = _ins_parts(case, rng)
    n, npe = mesh.n_nodes, mesh.npe
    conn, val, points = _geometry(mesh)
    x, phi, phid, fixed = _t(mesh.coords), _t(phi), torch.zeros(n, dtype=torch.float64, device=val.device), _t(wall, torch.long)
    iso2 = (_t(diff) ** 2).sum(1)
    am, af, ga, dt, t = prm["alpha_m"], prm["alpha_f"], prm["gamma"], prm["dt"], 0.0
    rows = conn[:, :, None].expand(-1, npe, npe).reshape(-1)
    cols = conn[:, None, :].expand(-1, npe, npe).reshape(-1)
    for _ in range(case["steps"]):
        s, c = torch.sin(math.pi * x), math.cos(math.pi * t / 8.0)
        vel = torch.stack([c * torch.sin(2 * math.pi * x[:, 1]) * s[:, 0] ** 2,
                           -c * torch.sin(2 * math.pi * x[:, 0]) * s[:, 1] ** 2, torch.zeros_like(phi)], 1)
        mat, rhs = 0.0, 0.0
        ve, pe, de = vel[conn], phi[conn], phid[conn]
        for g, (inv, dn, dv) in enumerate(points):
            m = (inv[:, :, :, None] * inv[:, :, None, :]).sum(1)
            u = (val[g][None, :, None] * ve).sum(1)
            tau = (4.0 / dt ** 2 + (u[:, :, None] * m * u[:, None, :]).sum((1, 2)) + iso2 * (m * m).sum((1, 2))).rsqrt()
            a = (dn * u[:, None, :]).sum(-1)
            left = (val[g][None, :] + tau[:, None] * a) * dv[:, None]
            mat = mat + left[:, :, None] * (am * val[g][None, None, :] + af * dt * ga * a[:, None, :])
            r = (1.0 - am) * (val[g][None, :] * de).sum(1) + (a * pe).sum(1) + af * dt * (1.0 - ga) * (a * de).sum(1)
            rhs = rhs - left * r[:, None]
        b = _node_sum(conn, rhs[..., None], n)[:, 0]
        b[fixed] = 0.0
        csr = torch.sparse_coo_tensor(torch.stack([rows, cols]), mat.reshape(-1), (n, n)).coalesce().to_sparse_csr()
        diag = torch.zeros(n, dtype=torch.float64, device=x.device).index_add_(
            0, conn.reshape(-1), mat.diagonal(dim1=1, dim2=2).reshape(-1))
        diag[fixed] = 1.0

        def times(v):
            y = (csr @ v[:, None])[:, 0]
            y[fixed] = v[fixed]
            return y

        new = _bicgstab(times, b, diag)
        phi = phi + dt * phid + ga * dt * (new - phid)
        phid = new
        t += dt
    return dict(phi=phi, phi_dot=phid, vel=vel)


def _bicgstab(times, b, diag):
    """A x = b to 1e-13 of |b|, Jacobi on the right."""
    x, r = torch.zeros_like(b), b.clone()
    shadow, p, rho, goal = r.clone(), r.clone(), r @ r, 1e-13 * b.norm()
    for _ in range(500):
        if r.norm() <= goal:
            break
        ph = p / diag
        v = times(ph)
        alpha = rho / (shadow @ v)
        s = r - alpha * v
        sh = s / diag
        t = times(sh)
        omega = (t @ s) / (t @ t)
        x = x + alpha * ph + omega * sh
        r = s - omega * t
        new = shadow @ r
        p = r + (new / rho) * (alpha / omega) * (p - omega * v)
        rho = new
    return x


def _ffd_exact(case, rng):
    (origin, n, s, t, u), nodes, vals, points = _ffd_parts(case, rng)
    axes = np.array([s, t, u])
    disp = np.zeros((n[0] * n[1] * n[2], 3))
    unit = axes / np.linalg.norm(axes, axis=1, keepdims=True)
    np.add.at(disp, nodes, vals @ unit)
    lattice = _t(disp.reshape(n[2], n[1], n[0], 3))
    out = []
    for part in _t(points).split(200_000):
        c = (part - _t(origin)) @ _t(np.linalg.inv(axes))
        inside = ((c >= 0.0) & (c <= 1.0)).all(1)
        bern = [torch.stack([math.comb(m - 1, i) * c[:, d] ** i * (1.0 - c[:, d]) ** (m - 1 - i) for i in range(m)], 1)
                for d, m in enumerate(n)]
        moved = torch.zeros_like(c)
        for z in range(n[2]):
            for y in range(n[1]):
                moved += (bern[2][:, z] * bern[1][:, y])[:, None] * (bern[0] @ lattice[z, y])
        out.append(torch.where(inside[:, None], moved, c))
    return torch.cat(out)


def exact(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "vms":
        out = _vms_exact(_vms_parts(case["nx"], case["ny"], case["nz"], case["flow"], rng, dual=case["dual"]),
                         case["steps"])
        return dict(out, norms=None) if case["norms"] else out
    if kind == "supg":
        return _supg_exact(_supg_parts(case["nx"], case["ny"], case["nz"], case["elem"], rng), case["steps"])
    if kind == "batch":
        return [_vms_exact((m, bc, dict(p, tot_dual_steps=0), s), case["steps"])["sol"]
                for m, bc, p, s in _batch_parts(case, rng)]
    if kind == "union":
        solve = _vms_exact if case["solver"] == "vms" else _supg_exact
        return [solve(p, case["steps"]) for p in _union_parts(case, rng)]
    return _ins_exact(case, rng) if kind == "ins" else _ffd_exact(case, rng)
