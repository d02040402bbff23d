"""Performance cases of the framework: what its users have it compute, through the public
entry points (SingleDimer, Program and the C ABI), over the range of sizes, numeric forms and
options that they use.

Kinds of case and the reference program each stands for:
  dimer     programs/single_dimer_pbc.f90: one collision cycle (n_md MD steps and a collision)
            of a batch of independent boxes, sampled after every cycle
  fluid     test/setup_simple_fluid.f90: one collision cycle of a plain SRD fluid
  sphere    test/setup_single_catalytic_fixed_sphere.f90: one collision cycle around a fixed
            catalytic sphere
  colloids  programs/n_colloids_pbc.f90: one collision cycle of many colloids, the production
            loop as a captured graph or the thermostat phase in the reference's call sequence
  step      a time step of a program of the user's own, written against the C ABI: streaming,
            grid shift, cell sort and one of the collisions (SRD with the bulk reaction,
            MPC-AT with the temperature, the wall collision of a channel flow)
  body      one MD step of a linked colloid of a few hundred beads (programs/single_body.f90):
            Verlet with iterative RATTLE on positions and velocities

A pass advances the state in place, as the programs do, and returns the state.
"""
import ctypes as C
import math
import random

import numpy as np
import torch

from rmpcdmd_amd import capi
from rmpcdmd_amd.programs import PROG_COLLOIDS, PROG_FLUID, PROG_SPHERE, Program
from rmpcdmd_amd.sim import SingleDimer
from rmpcdmd_amd.system import CellSet, ParticleSet

RHO = 10
FORMS = {"f64": capi.FP64, "f32": capi.FP32}
CHANNEL_G = 0.02  # acceleration of the channel flow
BODY_DT, BODY_PRECISION = 0.01, 1e-8


def listed():
    return [
        # the nanomotor in a small box, as a parameter scan runs it: 138,240 solvent
        # particles, bound by the latency of the MD steps
        {"name": "dimer_L24_f32", "kind": "dimer", "L": 24, "replicas": 1, "form": "f32", "lazy": 0},
        # the default box of the dimer program in the reference's precision
        {"name": "dimer_L48_f64", "kind": "dimer", "L": 48, "replicas": 1, "form": "f64", "lazy": 0},
        # the headline workload of the benchmark: 16 boxes of L = 64, 41.9 million particles
        {"name": "dimer_16xL64_f32", "kind": "dimer", "L": 64, "replicas": 16, "form": "f32", "lazy": 0},
        # a few boxes of an odd side with lazy streaming, the option for production runs
        {"name": "dimer_4xL45_f32_lazy", "kind": "dimer", "L": 45, "replicas": 4, "form": "f32", "lazy": 1},
        # the plain fluid at the driver's size and precision: small launches
        {"name": "fluid_L32_f64", "kind": "fluid", "Lx": 32, "Ly": 32, "Lz": 32, "form": "f64"},
        # a large fluid box: 21 million particles, bound by memory
        {"name": "fluid_L128_f32", "kind": "fluid", "Lx": 128, "Ly": 128, "Lz": 128, "form": "f32"},
        # the fixed catalytic sphere at the driver's size and precision
        {"name": "sphere_L32_f64", "kind": "sphere", "L": 32, "form": "f64"},
        # the colloidal suspension of the benchmark: 1000 colloids, 20.3 million particles
        {"name": "colloids_L128_f32", "kind": "colloids", "L": 128, "form": "f32", "graph": 1},
        # the thermostat phase that every suspension run begins with, in double precision
        {"name": "colloids_L48_f64_thermo", "kind": "colloids", "L": 48, "form": "f64", "graph": 0},
        # forced flow in a channel with ragged sides, in double precision
        {"name": "channel_60x31x45_f64", "kind": "step", "Lx": 60, "Ly": 31, "Lz": 45, "form": "f64", "collision": "wall"},
        # a thermostatted fluid at the benchmark's box size, with the temperature read back
        {"name": "thermo_L64_f32", "kind": "step", "Lx": 64, "Ly": 64, "Lz": 64, "form": "f32", "collision": "mpcat"},
        # the linked colloid of the benchmark: 300 beads, 1202 links
        {"name": "body_300", "kind": "body", "beads": 300},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dimer", "dimer", "fluid", "sphere", "colloids", "step", "step", "body"])
    form = rng.choice(["f32", "f64"])
    if kind == "dimer":
        L = rng.randint(16, 64)
        most = max(1, min(16, 16 * 64 ** 3 // (L ** 3 * (2 if form == "f64" else 1))))
        return {"kind": kind, "L": L, "replicas": _log_int(rng, 1, most), "form": form, "lazy": rng.choice([0, 0, 1])}
    if kind == "fluid":
        return {"kind": kind, **{k: _log_int(rng, 10, 112) for k in ("Lx", "Ly", "Lz")}, "form": form}
    if kind == "sphere":
        return {"kind": kind, "L": rng.randint(20, 48), "form": form}
    if kind == "colloids":
        graph = rng.choice([0, 1])
        return {"kind": kind, "L": rng.randint(32, 96 if graph else 56), "form": form, "graph": graph}
    if kind == "step":
        return {"kind": kind, **{k: _log_int(rng, 8, 90) for k in ("Lx", "Ly", "Lz")}, "form": form,
                "collision": rng.choice(["srd", "mpcat", "wall"])}
    return {"kind": kind, "beads": rng.randint(30, 500)}


# ---- the device-resident programs ------------------------------------------------------------
class _Raw:
    """device memory of a program's state, for torch.as_tensor; a tensor keeps this object, and
    with it the program whose memory it shows"""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": typestr, "version": 2}


def _view(owner, ptr, shape, typestr):
    return torch.as_tensor(_Raw(owner, ptr, shape, typestr), device="cuda")


def _particles(owner, p, names):
    real, small = ("<f8", "<i4") if p.form == capi.FP64 else ("<f4", "|u1")
    types = {"pos": real, "vel": real, "force": real, "image": "<i4", "id": "<i4", "species": small, "flags": small}
    n = p.n
    return {k: _view(owner, getattr(p, k), (3, n) if k in ("pos", "vel", "force", "image") else (n,), types[k])
            for k in names}


def _prepare_dimer(case, seed):
    L = case["L"]
    return {"sim": SingleDimer(L=(L, L, L), n_replicas=case["replicas"], form=FORMS[case["form"]], lazy=case["lazy"],
                               seed=seed), "replicas": case["replicas"]}


def _run_dimer(s):
    sim = s["sim"]
    sim.run(1)
    out = []
    # a replica's solvent and the first of them with its colloids: at most 64 arrays
    for r in range(s["replicas"]):
        sol, col, box, cells, st = sim.state(r)
        out.append(_particles(sim, sol, ("pos", "vel", "id") if r else ("pos", "vel", "id", "image", "species", "flags")))
        if r == 0:
            out.append(_particles(sim, col, ("pos", "vel", "force")))
    return out


def _prepare_program(case, seed):
    form = FORMS[case["form"]]
    if case["kind"] == "fluid":
        return {"prog": Program(PROG_FLUID, form=form, seed=seed, L=(case["Lx"], case["Ly"], case["Lz"]))}
    L = (case["L"],) * 3
    if case["kind"] == "sphere":
        return {"prog": Program(PROG_SPHERE, form=form, seed=seed, L=L)}
    # the suspension of n_colloids_pbc at its density, 1000 colloids at L = 128
    nc = max(2, int(1000 * case["L"] ** 3 / 128 ** 3))
    return {"prog": Program(PROG_COLLOIDS, form=form, seed=seed, L=L, n_colloids=nc, graph=case["graph"],
                            n_thermo=0 if case["graph"] else 1 << 30)}


def _run_program(s):
    prog = s["prog"]
    prog.run(1)
    sol, col, box, cells, st = prog.state()
    out = {"solvent": _particles(prog, sol, ("pos", "vel", "image", "id", "species", "flags")),
           "cell_count": _view(prog, cells.cell_count, (box.ncells,), "<i4"),
           "cell_start": _view(prog, cells.cell_start, (box.ncells,), "<i4")}
    if prog.kind != PROG_FLUID:
        out["temperature"] = float(st.temperature)
        out["colloids"] = _particles(prog, col, ("pos", "vel", "force"))
        out["n_extra_sorting"] = int(st.n_extra_sorting)
    return out


# ---- a program of the user's own on the C ABI ------------------------------------------------
STEP_TAU, STEP_T, STEP_RATE = 0.1, 1.0, 0.01


def _step_inputs(case, seed):
    """positions, velocities (FP64, rounded to the form when loaded), species of the solvent"""
    L = (case["Lx"], case["Ly"], case["Lz"])
    n = RHO * L[0] * L[1] * L[2]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    edges = torch.tensor(L, dtype=torch.float64, device="cuda")[:, None]
    pos = torch.rand(3, n, generator=gen, device="cuda", dtype=torch.float64) * edges * (1 - 2.0 ** -20)
    vel = torch.randn(3, n, generator=gen, device="cuda", dtype=torch.float64) * math.sqrt(STEP_T)
    vel -= vel.mean(dim=1, keepdim=True)
    species = 1 + (torch.rand(n, generator=gen, device="cuda") < 0.3).to(torch.int32)
    return L, n, pos, vel, species


def _prepare_step(case, seed):
    L, n, pos, vel, species = _step_inputs(case, seed)
    walls = case["collision"] == "wall"
    src, dst = ParticleSet(n, FORMS[case["form"]]), ParticleSet(n, FORMS[case["form"]])
    src.pos.copy_(pos)
    src.vel.copy_(vel)
    src.species.copy_(species)
    cs = CellSet(L, 1.0, walls)
    if walls:
        cs.box.bc[2] = capi.BOUNCE_BACK_BC
        for p in (src, dst):  # the flow's acceleration, as poiseuille_flow.f90 keeps it
            p.force[0] = CHANNEL_G
            p.force_old[0] = CHANNEL_G
    torch.cuda.synchronize()
    return {"src": src, "dst": dst, "cells": cs, "id_to_idx": torch.zeros(n, dtype=torch.int32, device="cuda"),
            "collision": case["collision"], "rng": random.Random(seed), "seed": seed, "step": 0,
            "wall_T": capi.d3([STEP_T, STEP_T, 0]), "wall_n": capi.i3([RHO, RHO, 0]), "te": C.c_double(0)}


def _run_step(s):
    src, dst, cs, k = s["src"], s["dst"], s["cells"], s["step"]
    box, cells = cs.boxp(), cs.cellsp()
    p = src.struct()
    if s["collision"] == "wall":
        capi.call("rmpcd_mpcd_stream_xforce_yzwall", box, p, STEP_TAU, CHANNEL_G)
        capi.call("rmpcd_md_vel", p, STEP_TAU)
        capi.call("rmpcd_apply_pbc", p, cs.box.edges)
    else:
        capi.call("rmpcd_mpcd_stream_periodic", box, p, STEP_TAU)
    capi.call("rmpcd_random_shift", box, capi.d3([s["rng"].random() for _ in range(3)]))
    q = dst.struct()
    capi.call("rmpcd_sort", box, p, q, C.c_void_p(s["id_to_idx"].data_ptr()), cells, 0)
    out = {}
    if s["collision"] == "wall":
        capi.call("rmpcd_wall_mpcd_step", box, cells, q, 1, s["wall_T"], s["wall_n"], 0, STEP_T, 1, 0, 0.0, None, None,
                  None, s["seed"], k)
    elif s["collision"] == "mpcat":
        capi.call("rmpcd_simple_mpcd_step", box, cells, q, None, s["seed"], k, 0, 0.0, 1, STEP_T, 1)
        capi.call("rmpcd_compute_temperature", box, cells, q, C.byref(s["te"]))
        out["temperature"] = float(s["te"].value)
    else:
        capi.call("rmpcd_simple_mpcd_step", box, cells, q, None, s["seed"], k, 0, 0.0, 0, STEP_T, 1)
        capi.call("rmpcd_bulk_reaction", box, cells, q, 2, 1, STEP_RATE, STEP_TAU, None, s["seed"], k)
    s["src"], s["dst"], s["step"] = dst, src, k + 1
    out.update(pos=dst.pos, vel=dst.vel, force=dst.force, image=dst.image, id=dst.id, species=dst.species,
               flags=dst.flags, id_to_idx=s["id_to_idx"], cell_count=cs.cell_count, cell_start=cs.cell_start)
    return out


# ---- a linked colloid ------------------------------------------------------------------------
BODY_EDGE = 40.0


def _body_inputs(case, seed):
    """beads on a Fibonacci sphere at the surface density of 300 beads on radius 4.5, linked
    to those closer than 1.8 mean spacings (i < j, by i then j)"""
    n = case["beads"]
    R = 4.5 * math.sqrt(n / 300)
    k = np.arange(n) + 0.5
    th, ph = np.arccos(1 - 2 * k / n), np.pi * (1 + 5 ** 0.5) * k
    r = R * np.stack([np.cos(ph) * np.sin(th), np.sin(ph) * np.sin(th), np.cos(th)], 1)
    i, j = np.triu_indices(n, 1)
    near = np.linalg.norm(r[i] - r[j], axis=1) < 1.8 * np.sqrt(4 * np.pi * R * R / n)
    links = np.ascontiguousarray(np.stack([i[near], j[near]], 1).astype(np.int32))
    dist = np.linalg.norm(r[links[:, 0]] - r[links[:, 1]], axis=1)
    rng = np.random.default_rng(seed)
    vel, force = rng.normal(size=(n, 3)), rng.normal(size=(n, 3))
    return n, links, dist, r + BODY_EDGE / 2, vel - vel.mean(0), force - force.mean(0)


def _prepare_body(case, seed):
    n, links, dist, pos, vel, force = _body_inputs(case, seed)
    p = ParticleSet(n, capi.FP64).load(pos=pos, vel=vel, force=force, force_old=force)
    torch.cuda.synchronize()
    return {"p": p, "links": links, "dist": dist, "pos_rattle": p.pos.clone(),
            "mass_each": torch.ones(n, dtype=torch.float64, device="cuda"), "mass": (C.c_double * 1)(1.0),
            "edges": capi.d3([BODY_EDGE] * 3), "it": C.c_int32(0)}


def _run_body(s):
    p = s["p"]
    h, links, dist = p.struct(), s["links"].ctypes.data_as(C.c_void_p), s["dist"].ctypes.data_as(C.c_void_p)
    mass_each, nl, it = C.c_void_p(s["mass_each"].data_ptr()), len(s["dist"]), C.byref(s["it"])
    s["pos_rattle"].copy_(p.pos)
    capi.call("rmpcd_colloid_md_pos", h, mass_each, BODY_DT)
    capi.call("rmpcd_rattle_body_pos", h, C.c_void_p(s["pos_rattle"].data_ptr()), links, dist, nl, s["mass"], 1,
              BODY_DT, s["edges"], BODY_PRECISION, it)
    capi.call("rmpcd_colloid_md_vel", h, mass_each, BODY_DT)
    capi.call("rmpcd_rattle_body_vel", h, links, dist, nl, s["mass"], 1, BODY_DT, s["edges"], BODY_PRECISION, it)
    return {"pos": p.pos, "vel": p.vel, "pos_rattle": s["pos_rattle"]}


def prepare(case, seed):
    if case["kind"] == "dimer":
        return {"run": _run_dimer, **_prepare_dimer(case, seed)}
    if case["kind"] == "step":
        return {"run": _run_step, **_prepare_step(case, seed)}
    if case["kind"] == "body":
        return {"run": _run_body, **_prepare_body(case, seed)}
    return {"run": _run_program, **_prepare_program(case, seed)}


def run(state):
    return state["run"](state)


def work(case):
    """Bytes and operations of one pass.  w is a real's size, S the state that a sort permutes
    (position, velocity, image, species, flags); 16 / rho are a cell's count and start, written
    and read.  Eager streaming moves 9 w per particle and MD step (read position and velocity,
    write the position); where particles are moved only when read, a cycle reads and writes
    the state once."""
    if case["kind"] == "body":
        n = case["beads"]
        return {"bytes": 8.0 * (6 + 3 + 6 + 3) * n, "flops": 60.0 * 4 * n}  # one sweep of about 4 n links
    w, S = (8, 68) if case["form"] == "f64" else (4, 38)
    flops = 60.0  # of a particle's collision and streaming
    if case["kind"] == "dimer":
        n = RHO * case["L"] ** 3 * case["replicas"]
        return {"bytes": float(n * ((0 if case["lazy"] else 50 * 9 * w) + 2 * S + 16 / RHO)), "flops": (flops + 6 * 50) * n}
    if case["kind"] == "fluid":
        n = RHO * case["Lx"] * case["Ly"] * case["Lz"]
        return {"bytes": float(n * (2 * (S + 4) + 16 / RHO)), "flops": flops * n}
    if case["kind"] == "sphere":  # ten eager MD steps and the collision
        n = RHO * case["L"] ** 3
        return {"bytes": float(n * (10 * 9 * w + 2 * (S + 4) + 16 / RHO)), "flops": (flops + 6 * 10) * n}
    if case["kind"] == "colloids":  # every particle once a cycle, those near a colloid (about 9 %) every step
        n = RHO * case["L"] ** 3
        return {"bytes": float(n * (0.09 * 50 * 9 * w + 2 * (S + 4) + 16 / RHO)), "flops": (flops + 6 * 50 * 0.09) * n}
    n = RHO * case["Lx"] * case["Ly"] * case["Lz"]
    # the sort also carries both forces and the id, and writes id_to_idx
    return {"bytes": float(n * (2 * (S + 6 * w + 4) + 4 + 16 / RHO)), "flops": flops * n}


# ---- the same in 64 bits, with torch and numpy alone -----------------------------------------
_SRD, _THERMO, _INIT, _SHIFT, _PLACE, _WALL = 1, 8, 6, 5, 7, 9  # second key words of the streams


def _threefry(c0, c1, k0, k1):
    """Threefry-2x64-20 (Salmon et al., SC'11) on int64 tensors, whose sums wrap"""
    def i64(v):
        v &= 2 ** 64 - 1
        return v - 2 ** 64 if v >= 2 ** 63 else v
    ks = [i64(k0), i64(k1), i64(0x1BD11BDAA9FC1A22 ^ (k0 & (2 ** 64 - 1)) ^ k1)]
    x0, x1 = c0 + ks[0], c1 + ks[1]
    for r in range(20):
        rot = (16, 42, 12, 31, 16, 32, 24, 21)[r & 7]
        x0 = x0 + x1
        x1 = ((x1 << rot) | ((x1 >> (64 - rot)) & ((1 << rot) - 1))) ^ x0
        if (r & 3) == 3:
            q = (r + 1) >> 2
            x0 = x0 + ks[q % 3]
            x1 = x1 + ks[(q + 1) % 3] + q
    return x0, x1


def _uniform(x):
    return ((x >> 11) & (2 ** 53 - 1)).double() * 2.0 ** -53


def _uniforms(step, item, seed, stream):
    a, b = _threefry(torch.full_like(item, step), item, seed, stream)
    return _uniform(a), _uniform(b)


def _normals(step, item, seed, stream):
    a, b = _uniforms(2 * step, item, seed, stream)
    c, d = _uniforms(2 * step + 1, item, seed, stream)
    r1, r2 = torch.sqrt(-2 * torch.log(1 - a)), torch.sqrt(-2 * torch.log(1 - c))
    return torch.stack([r1 * torch.cos(2 * math.pi * b), r1 * torch.sin(2 * math.pi * b), r2 * torch.cos(2 * math.pi * d)])


def _axes(step, cell, seed):
    """a unit vector for each cell by Marsaglia's method"""
    out = torch.zeros(3, cell.numel(), dtype=torch.float64, device=cell.device)
    todo, k = torch.arange(cell.numel(), device=cell.device), 0
    while todo.numel():
        a, b = _uniforms(step, cell[todo] + (k << 40), seed, _SRD)
        a, b = 2 * a - 1, 2 * b - 1
        s = a * a + b * b
        ok = s < 1
        f = 2 * torch.sqrt(1 - s[ok])
        out[:, todo[ok]] = torch.stack([a[ok] * f, b[ok] * f, 1 - 2 * s[ok]])
        todo, k = todo[~ok], k + 1
    return out


def _hilbert(p, M):
    """compact Hilbert index (Hamilton and Rau-Chaplin) of the integer points p (3 tensors)"""
    def ror(x, d):
        return ((x >> d) | (x << (3 - d))) & 7

    def rol(x, d):
        return ((x << d) | (x >> (3 - d))) & 7
    dev = p[0].device
    entry = torch.tensor([0, 0, 0, 3, 3, 6, 6, 5], device=dev)
    turn = torch.tensor([0, 1, 1, 2, 2, 1, 1, 0], device=dev)
    e = torch.zeros_like(p[0])
    d = torch.full_like(e, 2)
    h = torch.zeros_like(e)
    for i in reversed(range(max(M))):
        live = sum((M[k] > i) << k for k in range(3))
        r1 = (d + 1) % 3
        mask = ror(torch.full_like(e, live), r1)
        w = ror(sum(((p[k] >> i) & 1) << k for k in range(3)) ^ e, r1)
        w = w ^ (w >> 1) ^ (w >> 2)
        for k in (2, 1, 0):
            on = (mask >> k) & 1
            h = torch.where(on == 1, (h << 1) | ((w >> k) & 1), h)
        e = e ^ rol(entry[w], r1)
        d = (d + turn[w] + 1) % 3
    return h


def _sorted_cells(pos, L, origin, real, walls):
    """cell keys (in the precision of the positions), the stable order by key, counts"""
    M = [max(1, (v - 1).bit_length()) for v in L]
    p = []
    for k in range(3):
        c = torch.floor(pos[k].to(real) - torch.tensor(origin[k], dtype=real, device=pos.device)).long()
        p.append(c if walls and k == 2 else torch.where(c == L[k], torch.zeros_like(c), c))
    key = _hilbert(p, M)
    key, order = torch.sort(key, stable=True)
    nc = 1 << sum(M)
    z = p[2][order] & ((1 << M[2]) - 1)
    return key, order, torch.bincount(key, minlength=nc), z


def _cell_sums(key, nc, v):
    return torch.zeros(v.shape[0], nc, dtype=torch.float64, device=v.device).index_add_(1, key, v)


def _srd(vel, key, mean, axes):
    """rotation by -90 degrees about each cell's axis: n (n.w) - n x w"""
    u, n = mean[:, key], axes[:, key]
    w = vel - u
    return u + n * (n * w).sum(0) - torch.linalg.cross(n, w, dim=0)


def _fold(x, edges, image):
    for k in range(3):
        jump = torch.floor(x[k] / edges[k])
        image[k] += jump.long()
        x[k] = x[k] - jump * edges[k]


def _channel_flight(x0, v0, Lz, Ly, t, g):
    """a bounce-back flight between z walls with periodic y; a crossing of the y boundary on
    the way only counts an image, which is added back at the end"""
    tz = (Lz - x0[2]) / v0[2] if v0[2] > 0 else -x0[2] / v0[2]
    x = [x0[0] + v0[0] * tz + g * tz * tz / 2, x0[1] + v0[1] * tz, x0[2] + v0[2] * tz]
    v = [-(v0[0] + g * tz), -v0[1], -v0[2]]
    t -= tz
    return [x[0] + v[0] * t + g * t * t / 2, x[1] + v[1] * t, x[2] + v[2] * t], [v[0] + g * t, v[1], v[2]]


def _exact_step(case, seed):
    L, n, pos, vel, species = _step_inputs(case, seed)
    real = torch.float64 if case["form"] == "f64" else torch.float32
    pos, vel = pos.to(real), vel.to(real)
    walls = case["collision"] == "wall"
    image = torch.zeros(3, n, dtype=torch.long, device="cuda")
    force = torch.zeros(3, n, dtype=torch.float64, device="cuda")
    if walls:
        g, t = CHANNEL_G, STEP_TAU
        x0, v = pos.double(), vel.double()
        x = x0 + v * t
        x[0] += g * t * t / 2
        hit = torch.nonzero((x[2] < 0) | (x[2] > L[2]))[:, 0]
        if hit.numel() > 200000:
            return None
        flown = [_channel_flight(a, b, L[2], L[1], t, g) for a, b in zip(x0[:, hit].T.tolist(), v[:, hit].T.tolist())]
        force[0] = g
        moved = torch.ones(n, dtype=torch.bool, device="cuda")
        if flown:
            x[:, hit] = torch.tensor([f[0] for f in flown], dtype=torch.float64, device="cuda").T
            v[:, hit] = torch.tensor([f[1] for f in flown], dtype=torch.float64, device="cuda").T
            moved[hit] = False
        v[0] += torch.where(moved, g * t, 0.0)  # the others' velocities change in md_vel
        pos = x.to(real)
        _fold(pos, L, image)
        vel = v
    else:
        # the step's own rounding places the particles in cells
        pos = pos + vel * torch.tensor(STEP_TAU, dtype=real, device="cuda")
        _fold(pos, L, image)
        vel = vel.double()
    rng = random.Random(seed)
    origin = [rng.random() - 1 for _ in range(3)]
    key, order, count, z = _sorted_cells(pos, [L[0], L[1], L[2]], origin, real, walls)
    nc = count.numel()
    vel, pos = vel[:, order], pos[:, order]
    total, cells = _cell_sums(key, nc, vel), torch.arange(nc, device="cuda")
    out = {k: None for k in ("image", "id", "species", "flags", "id_to_idx", "cell_count", "cell_start")}
    many = (count > 1)[key]
    if case["collision"] == "mpcat":
        new = _normals(0, order, seed, _THERMO) * math.sqrt(STEP_T)
        new = new + ((total - _cell_sums(key, nc, new)) / count.clamp(min=1))[:, key]
        vel = torch.where(many, new, vel)
        d = vel - (_cell_sums(key, nc, vel) / count.clamp(min=1))[:, key]
        kin = _cell_sums(key, nc, (d * d).sum(0, keepdim=True))[0]
        ok = count > 1
        out["temperature"] = float((kin[ok] / (3 * (count[ok] - 1))).sum() / ok.sum())
    else:
        size = count.double()
        if walls:
            layer = torch.zeros(nc, dtype=torch.long, device="cuda")
            layer[key] = z
            extra = torch.where(((layer == 0) | (layer == L[2])) & (count > 0) & (count < RHO), RHO - count, 0)
            total = total + _normals(0, cells, seed, _WALL) * torch.sqrt(extra.double() * STEP_T)
            size = size + extra
        vel = torch.where(many, _srd(vel, key, total / size.clamp(min=1), _axes(0, cells, seed)), vel)
    out.update(pos=pos.double(), vel=vel, force=force)
    return out


def _exact_fluid(case, seed):
    """FP64 alone: in FP32 the rounding of the collision decides which cell a particle on a
    cell's edge streams into, and so the order of all that follow"""
    if case["form"] != "f64":
        return None
    L = (case["Lx"], case["Ly"], case["Lz"])
    n, T, tau = RHO * L[0] * L[1] * L[2], 1.0 / 3.0, 0.1
    item = torch.arange(n, device="cuda")
    vel = _normals(0, item, seed, _INIT) * math.sqrt(T)
    vel = vel - vel.sum(1, keepdim=True) / n
    a, b = _uniforms(0, item, seed, _PLACE)
    c, _ = _uniforms(0, item + (1 << 40), seed, _PLACE)
    pos = torch.stack([a * L[0], b * L[1], c * L[2]])

    def shift(s):
        zero = torch.zeros(1, dtype=torch.long)
        a, b = _uniforms(s, zero, seed, _SHIFT)
        c, _ = _uniforms(s, zero + 1, seed, _SHIFT)
        return [float(a) - 1, float(b) - 1, float(c) - 1]

    key, order, count, _ = _sorted_cells(pos, L, (0.0, 0.0, 0.0), torch.float64, False)
    pos, vel, nc = pos[:, order], vel[:, order], count.numel()
    mean = _cell_sums(key, nc, vel) / count.clamp(min=1)
    vel = torch.where((count > 1)[key], _srd(vel, key, mean, _axes(0, torch.arange(nc, device="cuda"), seed)), vel)
    pos = pos + vel * tau
    _fold(pos, L, torch.zeros(3, n, dtype=torch.long, device="cuda"))
    _, order, _, _ = _sorted_cells(pos, L, shift(1), torch.float64, False)
    solvent = {k: None for k in ("image", "id", "species", "flags")}
    return {"solvent": {**solvent, "pos": pos[:, order], "vel": vel[:, order]}, "cell_count": None, "cell_start": None}


def _exact_body(case, seed):
    """RATTLE is a Gauss-Seidel iteration over the links; in plain Python, so for small bodies"""
    if case["beads"] > 320:
        return None
    n, links, dist, pos0, vel0, force = _body_inputs(case, seed)
    dt, dist = BODY_DT, dist.tolist()
    links = [(int(a), int(b)) for a, b in links]
    pos = (pos0 + dt * vel0 + dt * dt * force / 2).tolist()
    vel, old = vel0.tolist(), pos0.tolist()
    la, lb = np.array([a for a, _ in links]), np.array([b for _, b in links])
    da = np.array(dist)
    for _ in range(1000):
        for (a, b), d in zip(links, dist):
            pa, pb, va, vb, ra, rb = pos[a], pos[b], vel[a], vel[b], old[a], old[b]
            r0, r1, r2 = ra[0] - rb[0], ra[1] - rb[1], ra[2] - rb[2]
            s0, s1, s2 = pa[0] - pb[0], pa[1] - pb[1], pa[2] - pb[2]
            rr, ss, rs = r0 * r0 + r1 * r1 + r2 * r2, s0 * s0 + s1 * s1 + s2 * s2, r0 * s0 + r1 * s1 + r2 * s2
            g = (rs - math.sqrt(rs * rs - rr * (ss - d * d))) / (dt * 2 * rr)
            for k, r in ((0, r0), (1, r1), (2, r2)):
                pa[k] -= g * dt * r
                pb[k] += g * dt * r
                va[k] -= g * r
                vb[k] += g * r
        x = np.array(pos)
        if np.abs(np.linalg.norm(x[la] - x[lb], axis=1) - da).max() < BODY_PRECISION:
            break
    x = np.array(pos)
    vel = (np.array(vel) + dt * force).tolist()
    seps = (x[la] - x[lb]).tolist()
    for _ in range(1000):
        for (a, b), s, d in zip(links, seps, dist):
            va, vb = vel[a], vel[b]
            k2 = ((va[0] - vb[0]) * s[0] + (va[1] - vb[1]) * s[1] + (va[2] - vb[2]) * s[2]) / (d * d * 2)
            for k in range(3):
                va[k] -= k2 * s[k]
                vb[k] += k2 * s[k]
        v = np.array(vel)
        worst = np.abs(((v[la] - v[lb]) * np.array(seps)).sum(1) / (da * da * 2)).max()
        if worst < BODY_PRECISION:
            break
    return {"pos": x.T, "vel": np.array(vel).T, "pos_rattle": pos0.T}


def exact(case, seed):
    """What the first pass returns, in 64 bits.  The dimer, sphere and colloid programs draw
    and equilibrate their own start; a value for them would be those programs again."""
    if case["kind"] == "step":
        return _exact_step(case, seed)
    if case["kind"] == "fluid":
        return _exact_fluid(case, seed)
    if case["kind"] == "body":
        return _exact_body(case, seed)
    return None
