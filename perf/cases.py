"""The work that users of this framework have it do, as cases that can be timed one by one.

A case is a dict of plain values. `listed()` gives the fixed ones, `draw(rng)` one more of the same ranges,
`prepare(case, seed)` what a program holds before the call (device meshes with a seeded state, options), `run(state)`
one pass through the public entry points, `work(case)` the bytes and operations the pass cannot do without, and
`exact(case, seed)` the result of the same pass in plain 64-bit torch.

The kinds of case:
  update   Solver::update, `steps` at a time: enqueued with the time step on the device (sync False), or one by one with
           the status read back (sync True)
  admis    what the reference's driver does each iteration without a smoothness indicator: set_art_visc_admis, update
  smooth   the same with one: update_art_visc_smoothness, update
  batch    one update of a group of independent boxes of several row sizes
  metrics  calc_jacobian of a deformed mesh, as after every change of the mesh
"""
import copy
import ctypes
import functools
import math
import random

import numpy as np
import torch

from hexed_amd import abi, configs, mesh
from hexed_amd.device import Context, Device_group, Device_mesh

GAMMA = 1.4
R_AIR = 287.05287
FORMS = {"fp64": abi.HX_FP64, "fp32_mfma": abi.HX_FP32_MFMA}

BASE = dict(kind="update", mesh="box", nd=3, rs=6, n=16, deformed=False, visc=False, form="fp64", steps=1, sync=False,
            local_time=False, use_filter=False, fix_admis=False, bc="freestream")


def _case(**kw):
    return {**BASE, **kw}


def listed():
    return [
        # a 2D Euler run on a small Cartesian mesh, one step per call, as a driver that reads every time step makes it
        _case(name="euler2d_16_sync", nd=2, n=16, sync=True),
        # a 2D Navier-Stokes run to a steady state between walls: local time stepping, the modal filter and the
        # admissibility check after every stage
        _case(name="ns2d_96_wall_fix", nd=2, n=96, deformed=True, visc=True, sync=True, local_time=True,
              use_filter=True, fix_admis=True, bc="no_slip"),
        # a 2D Navier-Stokes run of lower order in intervals of ten steps
        _case(name="ns2d_rs4_128", nd=2, rs=4, n=128, deformed=True, visc=True, steps=10),
        # 3D Euler on a uniform Cartesian mesh, the reference's arithmetic
        _case(name="euler_32", n=32),
        # the headline: 3D Navier-Stokes on a deformed mesh, in both arithmetic forms
        _case(name="ns_48", n=48, deformed=True, visc=True),
        _case(name="ns_48_fp32", n=48, deformed=True, visc=True, form="fp32_mfma"),
        # an odd mesh at an odd row size, stabilizing viscosity set before every step
        _case(name="ns_rs5_23_admis", kind="admis", rs=5, n=23, deformed=True, visc=True, sync=True, local_time=True),
        # the viscosity from the smoothness indicator before every step
        _case(name="ns_32_smooth", kind="smooth", n=32, deformed=True, visc=True, sync=True),
        # hanging faces: a 2:1-balanced tree, at the two row sizes such meshes are run with
        _case(name="tree_9", mesh="tree", n=9, steps=2),
        _case(name="tree_9_rs4", mesh="tree", n=9, rs=4, steps=5),
        # many small independent boxes of row sizes 4 to 6 in one group
        _case(name="batch_24_fp32", kind="batch", n=24, form="fp32_mfma", sync=True),
        # the metrics of a deformed mesh
        _case(name="metrics_32", kind="metrics", n=32, deformed=True),
    ]


def draw(rng):
    kind = rng.choice(["update"] * 6 + ["admis", "smooth", "batch", "metrics"])
    if kind == "batch":
        return _case(kind=kind, n=rng.randint(6, 28), form=rng.choice(["fp64", "fp32_mfma"]), sync=True)
    if kind == "update" and rng.random() < .25:
        return _case(mesh="tree", nd=3, rs=rng.randint(3, 7), n=rng.randint(4, 9), steps=rng.randint(1, 6),
                     sync=rng.random() < .3)
    nd = 3 if kind != "update" or rng.random() < .6 else 2
    rs = rng.randint(2, 8) if kind == "update" else rng.randint(3, 7)
    deformed = kind != "update" or rng.random() < .6
    visc = kind in ("admis", "smooth") or (deformed and rng.random() < .6)
    # from a few thousand points to a fifth of the largest listed mesh
    points = math.exp(rng.uniform(math.log(5e3), math.log(5e6)))
    n = max(3, round((points / rs ** nd) ** (1 / nd)))
    sync = kind != "update" or rng.random() < .4
    return _case(kind=kind, nd=nd, rs=rs, n=n, deformed=deformed, visc=visc, sync=sync,
                 steps=1 if sync or points > 1e6 else rng.randint(1, 10), local_time=rng.random() < .3,
                 use_filter=kind == "update" and rng.random() < .25,
                 form=rng.choice(["fp64", "fp64", "fp32_mfma"]) if kind == "update" else "fp64")


# ---- meshes -----------------------------------------------------------------------------------------------------------

def _key(case):
    return tuple(sorted((k, v) for k, v in case.items() if k != "name"))


def _flow(case):
    """(density, speed, pressure) of the freestream: air at Mach 0.3 and Re 1e4 on unit length, or unit density at Mach
    0.8."""
    if case["visc"]:
        rho, u, p, _ = configs.ns_freestream()
        return rho, u, p
    return 1., .8, 1 / GAMMA


def _freestream(case):
    rho, u, p = _flow(case)
    return configs.freestream_state(case["nd"], rho, [u] + [0.] * (case["nd"] - 1), p)


def _box(nd, rs, n, deformed, bc):
    """Connectivity of an n^nd box on the unit cube (elements, connections and slots ordered as `mesh.box` orders
    them) without its geometry, which a deformed mesh gets from calc_jacobian."""
    h, n_e = 1. / n, n ** nd
    grid = np.stack(np.unravel_index(np.arange(n_e), (n,) * nd), axis=1)
    con_a = [np.nonzero(grid[:, d] < n - 1)[0] for d in range(nd)]
    con_d = np.concatenate([np.full(len(a), d) for d, a in enumerate(con_a)])
    con_b = np.concatenate([a + n ** (nd - 1 - d) for d, a in enumerate(con_a)])
    con_a = np.concatenate(con_a)
    bnd = [(d, s, np.nonzero(grid[:, d] == (n - 1) * s)[0]) for d in range(nd) for s in (0, 1)]
    bnd_d, bnd_s = (np.concatenate([np.full(len(e), x[k]) for x in bnd for e in x[2:]]) for k in (0, 1))
    bnd_e = np.concatenate([e for _, _, e in bnd])
    n_int, n_bnd = len(con_a), len(bnd_e)
    c, off = int(deformed), n_int if deformed else 0
    m = mesh.HostMesh(nd, rs, 0 if deformed else n_e, n_e if deformed else 0, 2 * (n_int + n_bnd), 2 * (off + n_bnd),
                      0 if deformed else n_int, off + n_bnd)
    slots = np.arange(2 * (n_int + n_bnd), dtype=np.int32).reshape(-1, 2)
    m.face_slot[c][con_a, 2 * con_d + 1] = slots[:n_int, 0]
    m.face_slot[c][con_b, 2 * con_d] = slots[:n_int, 1]
    m.face_slot[c][bnd_e, 2 * bnd_d + bnd_s] = slots[n_int:, 0]
    m.con_slot[c][:n_int] = slots[:n_int]
    m.con_dir[c][:n_int] = np.array([mesh.pack_dir(d, d, 1, 0) for d in range(nd)])[con_d]
    m.con_slot[1][off:] = slots[n_int:]
    m.con_dir[1][off:] = [mesh.pack_dir(d, d, s, 1 - s) for d, s in zip(bnd_d, bnd_s)]
    m.con_nslot[:] = np.arange(2 * (off + n_bnd)).reshape(-1, 2)
    m.bc_con = np.arange(off, off + n_bnd, dtype=np.int32)
    m.bc_serial = np.zeros(n_bnd, np.int32)
    m.bcs = [bc]
    m.nom_size[c][:] = h
    m.n_vertex = (n + 1) ** nd
    corner = np.stack(np.unravel_index(np.arange(2 ** nd), (2,) * nd), axis=1)
    m.vertex_ids[c][:] = (grid[:, None] + corner) @ [(n + 1) ** (nd - 1 - d) for d in range(nd)]
    if deformed:
        m.face_nslot[con_a, 2 * con_d + 1] = m.con_nslot[:n_int, 0]
        m.face_nslot[con_b, 2 * con_d] = m.con_nslot[:n_int, 1]
        m.face_nslot[bnd_e, 2 * bnd_d + bnd_s] = m.con_nslot[n_int:, 0]
    else:
        m.normals[:] = np.repeat(np.eye(nd)[bnd_d], 2, axis=0)[:, :, None]
        m.vertex_tss[0][:] = h / nd
    m.qpos[c] = np.empty((n_e, nd, 0))  # (the states are formed on the GPU from the vertices)
    return m


def _batch_sizes(case):
    """(row size, elements per edge, Mach number) of each box of a batch: 512 to 4096 elements, log-uniform."""
    r = random.Random(case["n"])
    return [(r.choice([4, 5, 6]), round(math.exp(r.uniform(math.log(512), math.log(4096))) ** (1 / 3)),
             r.uniform(.3, .9)) for _ in range(case["n"])]


def _mach_state(mach):
    return configs.freestream_state(3, 1., [mach, 0., 0.], 1 / GAMMA)


@functools.lru_cache(maxsize=3)
def _topology(key):
    """The host mesh of a case, which does not depend on the seed; for a batch {row size: (mesh, its boxes)}."""
    case = dict(key)
    if case["kind"] == "batch":
        out = {}
        for rs in (4, 5, 6):
            boxes = [b for b in _batch_sizes(case) if b[0] == rs]
            if boxes:
                out[rs] = mesh.concat([_box(3, rs, n, False, (abi.HX_BC_FREESTREAM, _mach_state(mach)))
                                       for _, n, mach in boxes]), boxes
        return out
    fs = _freestream(case)
    if case["mesh"] == "tree":
        return configs.tree_mesh(case["n"], case["rs"], 3, .085, 0, case["nd"], (abi.HX_BC_FREESTREAM, fs))
    bc = (abi.HX_BC_FREESTREAM, fs)
    if case["bc"] == "no_slip":
        bc = (abi.HX_BC_NO_SLIP, fs, {"thermal": abi.HX_THERMAL_HEAT_FLUX})
    m = _box(case["nd"], case["rs"], case["n"], case["deformed"], bc)
    if case["visc"]:
        m.av = [np.zeros((k, 2, m.nq)) if k else None for k in m.n_elem]
    if case["kind"] == "smooth":
        m.enable_av_generator()
    return m


def _vertices(nd, n, deformed, seed):
    """Vertex positions [(n + 1)^nd][nd] of a box, the interior ones of a deformed one moved by up to 10% of the
    spacing."""
    v = np.stack(np.unravel_index(np.arange((n + 1) ** nd), (n + 1,) * nd), axis=1)
    pos = v / n
    if deformed:
        inside = np.all((v > 0) & (v < n), axis=1)
        pos[inside] += np.random.default_rng(seed).uniform(-.1 / n, .1 / n, (int(inside.sum()), nd))
    return pos


def _positions(rs, corners):
    """Quadrature point positions [n][nd][nq] of elements with the given corners [n][2^nd][nd], on the GPU."""
    nd = corners.shape[2]
    x = _basis(rs)["node"]
    p = torch.as_tensor(corners, device="cuda").reshape((-1,) + (2,) * nd + (nd,))
    w = torch.stack([1 - x, x], dim=1)
    for d in range(nd):
        p = torch.tensordot(p, w, dims=([1], [1]))  # the corner index of dimension d becomes the last point index
    return p.reshape(p.shape[0], nd, -1)


def _smooth(pos, rng, amplitude):
    """A sum of eight seeded sines per axis whose amplitudes add up to `amplitude`."""
    nd, modes = pos.shape[1], 8
    amp = [[rng.random() + .5 for _ in range(modes)] for _ in range(nd)]
    total = sum(map(sum, amp))
    out = torch.zeros_like(pos[:, 0])
    for d in range(nd):
        for k in range(modes):
            out += amplitude * amp[d][k] / total * torch.sin(2 * math.pi * ((k + 1) * pos[:, d] + rng.random()))
    return out


def _state(pos, flow, seed):
    """Conserved variables [n][nv][nq] of the freestream with 1% smooth perturbations of density and velocity."""
    rho0, u0, p = flow
    nd, rng = pos.shape[1], random.Random(seed)
    rho = rho0 * (1 + _smooth(pos, rng, .01))
    vel = [u0 * _smooth(pos, rng, .01) + (u0 if d == 0 else 0.) for d in range(nd)]
    return torch.stack([rho * v for v in vel] + [rho, p / (GAMMA - 1) + .5 * rho * sum(v * v for v in vel)], dim=1)


def _corners(case, seed):
    m = _topology(_key(case))
    c = int(case["deformed"])
    return _vertices(case["nd"], case["n"], case["deformed"], seed)[m.vertex_ids[c]]


def _initial(case, seed):
    """The initial state of each class of a case's mesh (for a batch {row size: state})."""
    if case["kind"] == "batch":
        out = {}
        for rs, (m, boxes) in _topology(_key(case)).items():
            parts = []
            for k, (_, n, mach) in enumerate(boxes):
                ids = _box(3, 2, n, False, (abi.HX_BC_FREESTREAM, _mach_state(mach))).vertex_ids[0]
                parts.append(_state(_positions(rs, _vertices(3, n, False, 0)[ids]), (1., mach, 1 / GAMMA),
                                    1000 * seed + 10 * k + rs))
            out[rs] = torch.cat(parts)
        return out
    if case["mesh"] == "tree":
        return _state(torch.as_tensor(_topology(_key(case)).qpos[0], device="cuda"), _flow(case), seed)
    return _state(_positions(case["rs"], _corners(case, seed)), _flow(case), seed)


def _bulk_av(case):
    """The constant bulk artificial viscosity of the Navier-Stokes cases [m^2/s]."""
    return 1e-3 if case["visc"] and case["kind"] != "smooth" else 0.


# ---- what a program holds, and one pass ---------------------------------------------------------------------------------

class _View:
    """A field of a device mesh as a CUDA array."""

    def __init__(self, dev, field, cls, shape):
        n, p = ctypes.c_size_t(), ctypes.c_void_p()
        dev.ctx.check(dev.lib.hx_mesh_device_ptr(dev.ptr, field, cls, ctypes.byref(p), ctypes.byref(n)))
        assert n.value == math.prod(shape)
        self.dev = dev
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f8", "data": (p.value, False), "version": 2}


def _field(dev, field, cls, *shape):
    return torch.as_tensor(_View(dev, field, cls, shape), device="cuda")


def _options(case):
    visc, cond = configs.sutherland_air() if case["visc"] else (None, None)
    return abi.update_options(max_safety=.5 if case["local_time"] else .7, local_time=case["local_time"],
                              use_filter=case["use_filter"], visc=visc, cond=cond, fix_admis=case["fix_admis"])


def prepare(case, seed):
    ctx = Context(0)
    s = {"case": case, "ctx": ctx, "options": _options(case)}
    if case["kind"] == "batch":
        s["devs"], s["state"], n_cases = [], {}, 0
        for (rs, (m, boxes)), init in zip(_topology(_key(case)).items(), _initial(case, seed).values()):
            dev = Device_mesh(ctx, m)
            view = _field(dev, abi.HX_FIELD_STATE, 0, m.n_elem[0], m.nv, m.nq)
            view.copy_(init)
            torch.cuda.synchronize()
            dev.set_precision(FORMS[case["form"]])
            dev.set_cases(len(boxes), m.case_id)
            dev.compute_write_face()
            s["devs"].append(dev)
            s["state"]["rs%d" % rs] = view
            n_cases += len(boxes)
        s["group"] = Device_group(ctx, s["devs"])
        s["status"] = (abi.hx_update_status * n_cases)()
        ctx.synchronize()
        return s
    m = copy.copy(_topology(_key(case)))
    c = int(case["deformed"])
    if case["deformed"]:
        m.def_vertex_pos = _corners(case, seed)
    dev = Device_mesh(ctx, m)
    s.update(dev=dev, host=m, status=abi.hx_update_status(), vertices=m.vertex_data())
    n, nd = m.n_elem[c], case["nd"]
    if case["kind"] == "metrics":
        s["out"] = {"metrics": _field(dev, abi.HX_FIELD_METRICS, 1, n, nd * nd + 1, m.nq),
                    "normals": _field(dev, abi.HX_FIELD_NORMALS, 0, m.normals.shape[0], nd, m.nfq),
                    "vertex_tss": _field(dev, abi.HX_FIELD_VERTEX_TSS, 1, n, m.nvert)}
        return s
    if case["deformed"]:
        dev.calc_jacobian(s["vertices"])
    s["out"] = {"state": _field(dev, abi.HX_FIELD_STATE, c, n, m.nv, m.nq)}
    s["out"]["state"].copy_(_initial(case, seed))
    if case["visc"]:
        s["out"]["av"] = _field(dev, abi.HX_FIELD_AV, c, n, 2, m.nq)
        s["out"]["av"][:, 0] = _bulk_av(case)
    rho, u, p = _flow(case)
    s["speed"] = u
    s["av_options"] = abi.av_options(.05, case["rs"], rho, p / (GAMMA - 1) + .5 * rho * u * u)
    torch.cuda.synchronize()
    dev.set_precision(FORMS[case["form"]])
    dev.compute_write_face()
    dev.prolong()
    ctx.synchronize()
    return s


def run(s):
    case = s["case"]
    if case["kind"] == "batch":
        s["group"].update(s["options"], s["status"])
        return {**s["state"], "dt": [t.time_step for t in s["status"]]}
    dev, out = s["dev"], dict(s["out"])
    if case["kind"] == "metrics":
        dev.calc_jacobian(s["vertices"])
        return out
    if case["kind"] == "admis":
        out["indicator"] = dev.set_art_visc_admis(s["speed"], s["vertices"])
    elif case["kind"] == "smooth":
        out["residual"] = dev.update_art_visc_smoothness(s["av_options"])
    if case["sync"]:
        for _ in range(case["steps"]):
            dev.update(s["options"], s["status"])
        out["dt"] = s["status"].time_step
    else:
        dev.update_async(s["options"], case["steps"])
    return out


# ---- what a pass cannot do without ----------------------------------------------------------------------------------------

def work(case):
    """Element data per point, in 64 bits: an update reads and writes the state in each of its two stages, writes and reads
    the residual cache between them, and reads the time step scale, the metrics of deformed elements and (the viscous
    stage) the viscosity coefficients; a convective stage cannot start before its neighbours' last one is done. Face data
    are made from the state and not counted. Operations: the row contractions and the point fluxes."""
    if case["kind"] == "batch":
        per = [work(_case(rs=rs, n=n)) for rs, n, _ in _batch_sizes(case)]
        return {k: sum(p[k] for p in per) for k in ("bytes", "flops")}
    nd, rs = case["nd"], case["rs"]
    nv, met = nd + 2, nd * nd + 1 if case["deformed"] else 0
    if case["mesh"] == "tree":
        m = _topology(_key(case))
        points, nfp = m.n_dof, 2 * nd / rs
    else:
        points, nfp = case["n"] ** nd * rs ** nd, 2 * nd / rs
    if case["kind"] == "metrics":  # positions of the corners in; metrics and face normals out
        return {"bytes": 8. * points * (met + nd * nfp + 2 ** nd * (nd + 1) / rs ** nd),
                "flops": points * (2. * rs * nd * nd + 2. * nfp * rs * nd * nd + 30 * nd)}
    row = 2. * rs + 4 + 4                     # one derivative value with its share of the lift
    flux = 8. * nv + 30 * nfp * nv            # the volume flux, and the numerical fluxes of the faces
    conv = nd * nv * row + nd * flux
    bytes_, flops = 2. * (3 * nv + 1 + met), 2 * conv
    if case["visc"]:
        bytes_ += 2
        flops += (nd * (nd if met else 1) + nd) * nv * row + 150
    bytes_, flops = bytes_ * case["steps"], flops * case["steps"]
    if case["kind"] == "admis":               # the density in, the coefficient out
        bytes_ += 2
        flops += 2. * nd * rs
    if case["kind"] == "smooth":              # two advection stages of rs scalars, one diffusion step of three, the projection
        bytes_ += 2 * (3 * rs + nd + 1 + met) + 2 * 3 * 2 + 2 + met + 3
        flops += 2 * nd * rs * row + 2 * nd * nd * 3 * row
    return {"bytes": 8. * points * bytes_, "flops": points * flops}


# ---- the same in plain torch ----------------------------------------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _basis(rs):
    """Gauss-Legendre nodes on [0, 1] with their derivative, boundary and lifting matrices, and the scheme's tabulated
    constants (modal filter, smallest eigenvalues)."""
    x, w = np.polynomial.legendre.leggauss(rs)
    x, w = (x + 1) / 2, w / 2
    bary = np.array([1 / np.prod([x[j] - x[k] for k in range(rs) if k != j]) for j in range(rs)])
    diff = np.zeros((rs, rs))
    for i in range(rs):
        for j in range(rs):
            if i != j:
                diff[i, j] = bary[j] / bary[i] / (x[i] - x[j])
        diff[i, i] = -diff[i].sum()
    bound = np.array([[bary[j] * np.prod([e - x[k] for k in range(rs) if k != j]) for j in range(rs)] for e in (0., 1.)])
    lift = np.stack([-bound[0] / w, bound[1] / w], axis=1)
    table = mesh.basis(rs)
    t = {"node": x, "diff": diff, "bound": bound, "lift": lift, "filter": table["filter"]}
    out = {k: torch.as_tensor(np.ascontiguousarray(v), device="cuda") for k, v in t.items()}
    out["eig"] = [float(e) for e in table["eigenvals"]]
    return out


def _along(mat, a, axis):
    """mat applied along `axis` of a."""
    return torch.movedim(torch.tensordot(a, mat, dims=([axis], [1])), -1, axis)


class _Box:
    """A box of elements as grid arrays: every field is [n]*nd + [rs]*nd, faces along d lack point dimension d."""

    def __init__(self, nd, rs, n, corners, deformed):
        self.nd, self.rs, self.n, self.h, self.deformed = nd, rs, n, 1. / n, deformed
        self.b = _basis(rs)
        self.shape = (n,) * nd + (rs,) * nd
        if not deformed:
            self.tss = torch.full((n ** nd, 2 ** nd), self.h / nd, device="cuda", dtype=torch.float64)
            return
        pos = [p.reshape(self.shape) for p in _positions(rs, corners).unbind(1)]
        J = [[self.D(pos[i], j) / self.h for j in range(nd)] for i in range(nd)]
        self.normal = [[self.cof(J, j, i) for j in range(nd)] for i in range(nd)]  # n_ij of reference direction i
        self.det = sum(J[0][c] * self.cof(J, 0, c) for c in range(nd))
        self.face_normal = []  # [d][j] at the n + 1 interfaces along d
        for d in range(nd):
            f = []
            for j in range(nd):
                lo, hi = (self.cof([[self.B(s, a, d) for a in row] for row in J], j, d) for s in (0, 1))
                a, z = self.cut(lo, d, 0, 1), self.cut(hi, d, n - 1, n)
                f.append(torch.cat([a, .5 * self.cut(hi, d, 0, n - 1) + .5 * self.cut(lo, d, 1, n), z], dim=d))
            self.face_normal.append(f)

        def at_vertices(a):
            for d in range(nd):
                a = _along(self.b["bound"], a, nd + d)
            return a.reshape(n ** nd, 2 ** nd)
        size = sum(sum(at_vertices(self.normal[i][j]) ** 2 for j in range(nd)).sqrt() for i in range(nd))
        own = self.h * at_vertices(self.det) / size
        # each vertex takes the smallest value of the elements that share it
        ids = np.stack(np.unravel_index(np.arange(n ** nd), (n,) * nd), axis=1)
        corner = np.stack(np.unravel_index(np.arange(2 ** nd), (2,) * nd), axis=1)
        ids = torch.as_tensor((ids[:, None] + corner) @ [(n + 1) ** (nd - 1 - d) for d in range(nd)], device="cuda")
        shared = torch.full(((n + 1) ** nd,), math.inf, device="cuda", dtype=torch.float64)
        shared.scatter_reduce_(0, ids.reshape(-1), own.reshape(-1), "amin")
        self.tss = shared[ids]

    def D(self, a, d):
        return _along(self.b["diff"], a, self.nd + d)

    def B(self, s, a, d):
        return torch.tensordot(a, self.b["bound"][s], dims=([self.nd + d], [0]))

    def cut(self, a, d, lo, hi):
        return a.narrow(d, lo, hi - lo)

    def cof(self, J, r, c):
        """Cofactor (r, c) of the matrix J."""
        if self.nd == 2:
            return (1 - 2 * ((r + c) % 2)) * J[1 - r][1 - c]
        r1, r2, c1, c2 = (r + 1) % 3, (r + 2) % 3, (c + 1) % 3, (c + 2) % 3
        return J[r1][c1] * J[r2][c2] - J[r1][c2] * J[r2][c1]

    def lift(self, jump, d):
        """Both faces' jumps lifted into the element along d."""
        ax = self.nd + d
        view = [1] * (2 * self.nd)
        view[ax] = self.rs
        return sum(self.b["lift"][:, s].reshape(view) * jump[s].unsqueeze(ax) for s in (0, 1))

    def sides(self, a, d, ghost=None):
        """The two states at the interfaces along d: left elements' face 1, right elements' face 0; outside the ghost
        value, or the inside state again."""
        lo, hi = self.B(0, a, d), self.B(1, a, d)
        first, last = self.cut(lo, d, 0, 1), self.cut(hi, d, self.n - 1, self.n)
        if ghost is not None:
            first, last = torch.full_like(first, ghost), torch.full_like(last, ghost)
        return torch.cat([first, hi], dim=d), torch.cat([lo, last], dim=d)

    def normals(self, d, where):
        if self.deformed:
            return (self.normal if where == "volume" else self.face_normal)[d]
        return [1. if j == d else 0. for j in range(self.nd)]

    def conv_flux(self, u, nrm):
        nd = self.nd
        kin = .5 * sum(m * m for m in u[:nd]) / u[nd]
        p = (GAMMA - 1) * (u[nd + 1] - kin)
        mass = sum(m * k for m, k in zip(u, nrm))
        vol = mass / u[nd]
        return [u[j] * vol + p * nrm[j] for j in range(nd)] + [mass, (u[nd + 1] + p) * vol]

    def speed(self, u):
        nd = self.nd
        return (GAMMA * (GAMMA - 1) * u[nd + 1] / u[nd]).sqrt() + sum(m * m for m in u[:nd]).sqrt() / u[nd]

    def numerical(self, u, ghost, d):
        """The numerical flux at the interfaces along d, and the average of both states."""
        two = [self.sides(a, d, g) for a, g in zip(u, ghost)]
        left, right = [t[0] for t in two], [t[1] for t in two]
        nrm = self.normals(d, "face")
        c = torch.maximum(self.speed(left), self.speed(right)) * (sum(k * k for k in nrm) ** .5)
        f = [.5 * (a + b + c * (x - y)) for a, b, x, y in
             zip(self.conv_flux(left, nrm), self.conv_flux(right, nrm), left, right)]
        return f, [.5 * (x + y) for x, y in zip(left, right)]

    def pair(self, a, d):
        """An interface array as each element's (face 0, face 1) values along d."""
        return self.cut(a, d, 0, self.n), self.cut(a, d, 1, self.n + 1)

    def derivative(self, x, face, d):
        f = self.pair(face, d)
        return self.D(x, d) + self.lift([f[s] - self.B(s, x, d) for s in (0, 1)], d)

    def conv_rate(self, u, ghost):
        rate = [0.] * len(u)
        averages = []
        for d in range(self.nd):
            num, avg = self.numerical(u, ghost, d)
            averages.append(avg)
            vol = self.conv_flux(u, self.normals(d, "volume"))
            rate = [r - self.derivative(x, f, d) for r, x, f in zip(rate, vol, num)]
        return rate, averages

    def filtered(self, rate, use):
        if use:
            for d in range(self.nd):
                rate = [_along(self.b["filter"], r, self.nd + d) for r in rate]
        return rate


def _sutherland(t, ref, temp, off):
    return ref * (t / temp) ** 1.5 * (temp + off) / (t + off)


def _transport(u, nd):
    kin = .5 * sum(m * m for m in u[:nd]) / u[nd]
    temp = torch.clamp((u[nd + 1] - kin) / u[nd], min=0.) * (GAMMA - 1) / R_AIR
    return _sutherland(temp, 1.716e-5, 273., 111.), _sutherland(temp, .0241, 273., 194.) * (GAMMA - 1) / R_AIR


def _visc_flux(u, grad, bulk, nd):
    """f[v][j] from the gradients grad[v][j]."""
    mu, cond = _transport(u, nd)
    vel = [m / u[nd] for m in u[:nd]]
    vg = [[(grad[i][j] - vel[i] * grad[nd][j]) / u[nd] for j in range(nd)] for i in range(nd)]
    dil = (bulk * u[nd] - 2. / 3. * mu) * sum(vg[i][i] for i in range(nd))
    f = [[None] * nd for _ in range(nd + 2)]
    for j in range(nd):
        stress = [mu * (vg[i][j] + vg[j][i]) + (dil if i == j else 0.) for i in range(nd)]
        energy = grad[nd + 1][j] / u[nd] - u[nd + 1] / u[nd] ** 2 * grad[nd][j] - sum(v * g[j] for v, g in zip(vel, vg))
        for i in range(nd):
            f[i][j] = -stress[i]
        f[nd][j] = torch.zeros_like(mu)
        f[nd + 1][j] = -(sum(v * t for v, t in zip(vel, stress)) + cond * energy)
    return f


def _exact_update(case, box, init, ghost, bulk):
    """`steps` updates of a box with freestream ghosts: (state [n][nv][nq], last time step)."""
    nd, rs, h = box.nd, box.rs, box.h
    u = [a.reshape(box.shape) for a in init.unbind(1)]
    safety, cheby = (.5 if case["local_time"] else .7), 1 / (1 - math.cos(.5 * math.pi))
    cc, cd = -2 * .9 / box.b["eig"][0] * safety / cheby, -2 / box.b["eig"][1] * safety
    spacing = box.tss.reshape((-1,) + (2,) * nd)
    for _ in range(nd):  # the vertex spacing interpolated to the points
        spacing = torch.tensordot(spacing, torch.stack([1 - box.b["node"], box.b["node"]], dim=1), dims=([1], [1]))
    spacing = spacing.reshape(box.shape)
    det = box.det if box.deformed else 1.
    use = case["use_filter"]
    dt = 0.
    for _ in range(case["steps"]):
        scale = box.speed(u) / cc / spacing
        if case["visc"]:
            mu, cond = _transport(u, nd)
            scale = scale + torch.maximum(bulk + mu / u[nd], cond / u[nd]) / cd / spacing ** 2
        dt = cheby if case["local_time"] else float((1 / scale).min()) * cheby
        step = dt * (1 / scale if case["local_time"] else 1.) / h / det
        rate, avg = box.conv_rate(u, ghost)
        rate = first = box.filtered(rate, use)
        if case["visc"]:
            grad = [[None] * nd for _ in u]
            for v, a in enumerate(u):
                for j in range(nd):
                    g = 0.
                    for i in range(nd) if box.deformed else (j,):
                        nv, nf = (box.normals(i, w)[j] for w in ("volume", "face"))
                        g = g + box.derivative(a * nv, avg[i][v] * nf, i)
                    grad[v][j] = g / h / det
            f = _visc_flux(u, grad, bulk, nd)
            del grad
            visc, back = [], []
            for v in range(nd + 2):
                r = b = 0.
                for i in range(nd):
                    fi = sum(f[v][j] * box.normal[i][j] for j in range(nd)) if box.deformed else f[v][i]
                    r = r - box.D(fi, i)
                    left, right = box.sides(fi, i)
                    mean = box.pair(.5 * (left + right), i)
                    b = b - box.lift([mean[s] - box.B(s, fi, i) for s in (0, 1)], i)
                visc.append(r)
                back.append(b)
            visc, back = box.filtered(visc, use), box.filtered(back, use)
            rate = [a + b + c for a, b, c in zip(rate, visc, back)]
        u = [a + step * r for a, r in zip(u, rate)]
        second, _ = box.conv_rate(u, ghost)
        second = box.filtered(second, use)
        u = [a + step * (.5 / .9) * (r - q) for a, r, q in zip(u, second, first)]
    return torch.stack([a.reshape(-1, rs ** nd) for a in u], dim=1), dt


def exact(case, seed):
    if case["kind"] == "batch":
        out, dts = {}, []
        for (rs, (m, boxes)), init in zip(_topology(_key(case)).items(), _initial(case, seed).values()):
            parts, at = [], 0
            for _, n, mach in boxes:
                u, dt = _exact_update(case, _Box(3, rs, n, None, False), init[at:at + n ** 3], _mach_state(mach), 0.)
                parts.append(u)
                dts.append(dt)
                at += n ** 3
            out["rs%d" % rs] = torch.cat(parts)
        return {**out, "dt": dts}
    if case["kind"] in ("admis", "smooth") or case["mesh"] == "tree" or case["bc"] != "freestream":
        return None
    nd, rs, n = case["nd"], case["rs"], case["n"]
    box = _Box(nd, rs, n, _corners(case, seed), case["deformed"])
    if case["kind"] == "metrics":
        met = torch.stack([a.reshape(n ** nd, -1) for row in box.normal for a in row] + [box.det.reshape(n ** nd, -1)], dim=1)
        inner, outer = [], []
        for d in range(nd):
            f = torch.stack(box.face_normal[d], dim=nd)  # [n]*nd (n + 1 along d), nd, face points
            flat = lambda lo, hi: box.cut(f, d, lo, hi).reshape(-1, nd, rs ** (nd - 1))  # noqa: E731
            inner.append(flat(1, n))
            outer += [flat(0, 1), flat(n, n + 1)]
        nrm = torch.repeat_interleave(torch.cat(inner + outer), 2, dim=0)
        return {"metrics": met, "normals": nrm, "vertex_tss": box.tss}
    state, dt = _exact_update(case, box, _initial(case, seed), _freestream(case), _bulk_av(case))
    out = {"state": state}
    if case["visc"]:
        out["av"] = None
    if case["sync"]:
        out["dt"] = dt
    return out
