"""Timed work of the framework, as a user's program has it do it.

Six kinds of pass, each through public entry points:

  uniform     macro steps of one uniform case resident in HBM (gpu.GpuCase.advance):
              time step, three RK stages, halo fills.  The main path.
  serve       a batch of small independent cases through one ensemble: admitted,
              stepped with polls, read back, released.
  multilevel  one macro step of the multiresolution driver with local time
              stepping and remeshing (multilevel.MultiLevelSolver.advance).
  mr          the multiresolution operators of one level: children averaged into
              parents, wavelet details and decisions, refinement, jump halos.
  rhs         the per-block right-hand side a host code calls for its own blocks
              (alpaca_right_hand_side).
  level       the level-wise integration of a stage: boundary-flux right-hand
              side of listed leaves, buffer preparation, integration, halos.

Sizes are the repository's own (the 256^3 and 2D 128^2 configurations of bench.py,
its batched and multi-level legs, the grids of its tests) and odd ones between.
"""
import ctypes
import math
import random

import numpy as np
import torch

from alpaca_amd import cases as states
from alpaca_amd import ensemble, gpu, lts, multilevel
from alpaca_amd import multiresolution as mr

DEV = "cuda" if torch.cuda.is_available() else "cpu"
IC, HS, TC = gpu.IC, gpu.HS, gpu.TC
FLUX = {"hllc": gpu.FLUX_HLLC, "roe": gpu.FLUX_ROE}
FORM = {"fp64": gpu.FP64, "mixed": gpu.MIXED, "fma": gpu.FP64_FMA}
BC = {"z": gpu.BC_ZERO_GRADIENT, "p": gpu.BC_PERIODIC, "s": gpu.BC_SYMMETRY}
# Algorithmic FLOP per cell and RK stage (dimension, flux family) and per cell face.
FLOP_STAGE = {(3, "hllc"): 4549.0, (3, "roe"): 6109.0, (2, "hllc"): 2257.0, (2, "roe"): 2863.0}


def _uniform(name, dim, nb, bc, flux, form, steps, gamma=1.4, b=0.0):
    nb = list(nb) + [1] * (3 - len(nb))
    return {"name": name, "kind": "uniform", "dim": dim, "nx": nb[0], "ny": nb[1], "nz": nb[2],
            "bc": bc, "flux": flux, "form": form, "steps": steps, "gamma": gamma, "b": b}


def listed():
    return [
        # The smallest whole run: 2D 128^2 to an end time, advanced in chunks of steps
        # between two looks at the clock; launches and latency count.
        _uniform("2d-128-hllc", 2, (8, 8), "zz", "hllc", "fp64", 8),
        # A 2D channel of odd extents, symmetry walls, Roe, the mixed form.
        _uniform("2d-odd-roe-mixed", 2, (45, 23), "ps", "roe", "mixed", 2, gamma=1.32),
        # One large 2D case.
        _uniform("2d-2048-hllc", 2, (128, 128), "zz", "hllc", "fp64", 1),
        # The size of the reference's 3D test inputs: a handful of blocks, three kinds of side.
        _uniform("3d-small-roe", 3, (4, 2, 3), "zsp", "roe", "fp64", 2),
        # The headline configuration, in the bit-exact form: the largest.
        _uniform("3d-256-hllc", 3, (16, 16, 16), "ppp", "hllc", "fp64", 1),
        # The same problem a user runs with the other flux family at an eighth of the cells.
        _uniform("3d-128-roe", 3, (8, 8, 8), "ppp", "roe", "fp64", 1),
        # A liquid (stiffened gas) in an odd box in the contracted form.
        _uniform("3d-odd-hllc-fma", 3, (7, 5, 11), "zps", "hllc", "fma", 2, gamma=4.4, b=0.5),
        # The mixed form on 128^3.
        _uniform("3d-128-hllc-mixed", 3, (8, 8, 8), "ppp", "hllc", "mixed", 1),
        # A serving batch: 12 uneven 2D cases, FP64 and mixed in turn.
        {"name": "serve-12", "kind": "serve", "cases": 12, "steps": 32, "most": 12, "flux": "hllc"},
        # The multi-level mode of the benchmark: 4^3 level-0 nodes, maximum level 2.
        {"name": "multilevel-3d", "kind": "multilevel", "dim": 3, "n0": 4, "lmax": 2, "flux": "hllc"},
        # The operators between 160 parents and their children (every micro step of a
        # 3D run of this size).
        {"name": "mr-160", "kind": "mr", "dim": 3, "parents": 160},
        # A host code that hands over a few of its own blocks.
        {"name": "rhs-6", "kind": "rhs", "dim": 3, "blocks": 6, "flux": "hllc", "form": "fp64"},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["uniform"] * 6 + ["serve", "multilevel", "mr", "rhs", "rhs", "level"])
    flux = rng.choice(["hllc", "hllc", "roe"])
    form = rng.choice(["fp64", "fp64", "fma", "mixed"])
    if kind == "uniform":
        dim = rng.choice([2, 3])
        if dim == 2:
            blocks = _log(rng, 6, 9000)
            nx = max(1, min(blocks, int(round(math.sqrt(blocks) * math.exp(rng.uniform(-0.7, 0.7))))))
            nb = (nx, max(1, blocks // nx))
        else:
            blocks = _log(rng, 4, 2600 if flux == "hllc" else 1500)
            side = blocks ** (1.0 / 3.0)
            nx = max(1, int(round(side * math.exp(rng.uniform(-0.5, 0.5)))))
            ny = max(1, int(round(side * math.exp(rng.uniform(-0.4, 0.4)))))
            nb = (nx, ny, max(1, blocks // (nx * ny)))
        steps = 1 if blocks > 300 else rng.randint(1, 8 if dim == 2 else 3)
        c = _uniform("", dim, nb, "".join(rng.choice("zps") for _ in range(dim)), flux, form, steps,
                     gamma=round(rng.uniform(1.2, 1.67), 3), b=rng.choice([0.0, 0.0, 0.25]))
        del c["name"]
        return c
    if kind == "serve":
        return {"kind": "serve", "cases": rng.randint(4, 14), "steps": 8 * rng.randint(2, 4),
                "most": rng.randint(3, 12), "flux": flux}
    if kind == "multilevel":
        if rng.random() < 0.5:
            return {"kind": "multilevel", "dim": 2, "n0": rng.randint(2, 6), "lmax": rng.randint(1, 3),
                    "flux": flux}
        return {"kind": "multilevel", "dim": 3, "n0": rng.randint(2, 3), "lmax": rng.randint(1, 2),
                "flux": flux}
    if kind == "mr":
        dim = rng.choice([2, 3, 3])
        return {"kind": "mr", "dim": dim, "parents": _log(rng, 3, 220 if dim == 3 else 3000)}
    if kind == "rhs":
        dim = rng.choice([2, 3, 3])
        return {"kind": "rhs", "dim": dim, "blocks": _log(rng, 1, 900 if dim == 3 else 6000),
                "flux": flux, "form": form}
    dim = rng.choice([2, 3, 3])
    return {"kind": "level", "dim": dim, "blocks": _log(rng, 5, 1200 if dim == 3 else 8000),
            "flux": flux, "form": form}


# ------------------------------------------------------------------- inputs

def _field(dim, n, seed, gamma, b):
    """Domain conservatives [NE][nx][ny][nz]: a background with four constant
    quarters (contacts, shocks and shear between them), Gaussian blobs of density
    and pressure, and a smooth velocity."""
    r = random.Random(seed * 7919 + dim)
    n = list(n)[:dim]
    longest = max(n)
    x = [((torch.arange(m, dtype=torch.float64, device=DEV) + 0.5) / longest).reshape(
        [-1 if a == d else 1 for a in range(dim)]) for d, m in enumerate(n)]
    hi = [x[0] >= 0.5 * n[0] / longest, x[1] >= 0.5 * n[1] / longest]
    q = [(r.uniform(0.5, 1.5), r.uniform(0.5, 1.5), [r.uniform(-0.5, 0.5) for _ in range(dim)])
         for _ in range(4)]
    which = (hi[0].long() + 2 * hi[1].long()).expand(n)
    tab = torch.tensor([[s[0], s[1], *s[2]] for s in q], dtype=torch.float64, device=DEV)
    rho, p = tab[:, 0][which], tab[:, 1][which]
    vel = [tab[:, 2 + d][which] for d in range(dim)]
    for _ in range(6):
        width = r.uniform(0.04, 0.12)
        g = r.uniform(0.2, 2.0)
        for d in range(dim):
            c = r.uniform(0.0, n[d] / longest)
            g = g * torch.exp(-((x[d] - c) ** 2) / (2 * width * width))
        rho, p = rho + g, p + g * r.uniform(0.5, 1.5)
    for d in range(dim):
        k = r.randint(1, 3)
        vel[d] = vel[d] + 0.2 * torch.sin(2 * math.pi * k * x[(d + 1) % dim] + r.uniform(0, 6))
    e = (p + gamma * b) / (gamma - 1.0) + 0.5 * rho * sum(v * v for v in vel)
    u = torch.stack([rho, e] + [rho * v for v in vel])
    return u if dim == 3 else u[..., None]


def _haloed(dim, count, seed, gamma=1.4, b=0.0):
    """`count` haloed blocks [count][NE][24][24][24|1] cut out of one field."""
    per = max(1, int(math.ceil(count ** (1.0 / dim))))
    u = _field(dim, [per * 8 + 16] * dim, seed, gamma, b)
    if dim == 2:
        u = u[..., 0]
    w = u
    for a in range(dim):
        w = w.unfold(1 + a, TC, 8)
    order = list(range(1, 1 + dim)) + [0] + list(range(1 + dim, 1 + 2 * dim))
    w = w.permute(order).reshape((-1, dim + 2) + (TC,) * dim)[:count].contiguous()
    return w if dim == 3 else w[..., None].contiguous()


def _nb(case):
    return [case["nx"], case["ny"], case["nz"]][:case["dim"]]


def _desc(case):
    return gpu.make_desc(case["dim"], _nb(case), [BC[c] for c in case["bc"]], flux=FLUX[case["flux"]],
                         precision=FORM[case["form"]], gamma=case["gamma"], b=case["b"])


CFL = 0.5


def _serve_specs(case, seed):
    r, sizes = random.Random(seed * 104729 + 1), random.Random(case["cases"] * 64 + case["most"])
    out = []
    for i in range(case["cases"]):
        nx, ny = sizes.randint(2, case["most"]), sizes.randint(2, case["most"])
        out.append({"dim": 2, "nx": nx, "ny": ny, "nz": 1, "bc": "zz", "flux": case["flux"],
                    "form": ("fp64", "mixed")[i % 2], "gamma": r.uniform(1.2, 1.67), "b": 0.0,
                    "seed": r.randrange(1 << 30)})
    return out


def _ml_initial(dim, node, length, seed, gamma=1.4):
    """Conservatives of a node's internal cells: a dense hot ball and a ring of
    another density in a uniform stream."""
    r = random.Random(seed * 31 + 5)
    centre = [length * r.uniform(0.3, 0.7) for _ in range(dim)]
    radius2 = (length * r.uniform(0.12, 0.16)) ** 2
    jump = r.uniform(1.5, 2.5)
    flow = [r.uniform(0.2, 0.6) for _ in range(dim)]

    def initial(level, key):
        dx = node / (1 << level) / IC
        ax = [(key[a + 1] * IC + np.arange(IC) + 0.5) * dx for a in range(dim)]
        g = np.meshgrid(*ax, indexing="ij")
        inside = sum((g[a] - centre[a]) ** 2 for a in range(dim)) < radius2
        rho, p = 1.0 + jump * inside, 1.0 + 2.0 * jump * inside
        vel = [flow[a] * np.ones_like(rho) for a in range(dim)]
        c = states.primes_to_conservatives(dim, gamma, 0.0, rho, vel, p)
        return c[..., None] if dim == 2 else c
    return initial


def _mr_rows(case):
    """Pool layout: parents, their children, and the new children of a quarter of
    those; links of both, and the (link, location) pairs of jump halos."""
    kids = 1 << case["dim"]
    p = case["parents"]
    rows = [(p + i * kids + c, i, c, 1) for i in range(p) for c in range(kids)]
    base = p + p * kids
    parents = list(range(p, base, 4))
    fine = [(base + i * kids + c, s, c, 2) for i, s in enumerate(parents) for c in range(kids)]
    locations = multilevel.halo_locations(case["dim"])
    jumps = [(r, locations[(i * 5 + k) % len(locations)]) for i, r in enumerate(fine) for k in (0, 3)]
    return rows, fine, jumps, base + len(fine)


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def prepare(case, seed):
    kind = case["kind"]
    if kind == "uniform":
        u = _field(case["dim"], [m * IC for m in _nb(case)], seed, case["gamma"], case["b"])
        return {"case": gpu.GpuCase(_desc(case), u, CFL), "kind": kind, "steps": case["steps"]}
    if kind == "serve":
        specs = _serve_specs(case, seed)
        blocks = sum(s["nx"] * s["ny"] for s in specs)
        ens = ensemble.Ensemble(2, blocks, len(specs), [(FLUX[case["flux"]], gpu.FP64),
                                                       (FLUX[case["flux"]], gpu.MIXED)])
        return {"kind": kind, "ens": ens, "steps": case["steps"],
                "cases": [(_desc(s), _field(2, [s["nx"] * IC, s["ny"] * IC], s["seed"], s["gamma"], 0.0))
                          for s in specs]}
    if kind == "multilevel":
        dim, n0, lmax = case["dim"], case["n0"], case["lmax"]
        node = 1.0 / n0
        nodes = sum((n0 << level) ** dim for level in range(lmax + 1))
        be = multilevel.GpuBackend(dim, nodes, flux=FLUX[case["flux"]])
        sol = multilevel.MultiLevelSolver(be, dim, [n0] * dim, node, lmax, [gpu.BC_PERIODIC] * (2 * dim),
                                          _ml_initial(dim, node, 1.0, seed), CFL, 1e6, 1e-3, lmax,
                                          flux=FLUX[case["flux"]])
        sol.create_new_simulation()
        return {"kind": kind, "sol": sol}
    if kind == "mr":
        dim = case["dim"]
        rows, fine, jumps, n = _mr_rows(case)
        as_links = lambda x: torch.as_tensor(mr.make_links(x), device=DEV)  # noqa: E731
        return {"kind": kind, "dim": dim, "blocks": _haloed(dim, n, seed),
                "op": mr.Multiresolution(mr.ThresholdComputer(dim, 2, 2, 1e-2)),
                "links": as_links(rows), "fine": as_links(fine),
                "jumps": as_links([j[0] for j in jumps]),
                "where": torch.tensor([j[1] for j in jumps], dtype=torch.int32, device=DEV)}
    if kind == "rhs":
        dim, n = case["dim"], case["blocks"]
        desc = gpu.make_desc(dim, [n] + [1] * (dim - 1), [gpu.BC_ZERO_GRADIENT] * dim,
                             flux=FLUX[case["flux"]], precision=FORM[case["form"]], cell_size=1.0 / 64)
        avg = _haloed(dim, n, seed)
        return {"kind": kind, "desc": desc, "n": n, "avg": avg, "rhs": torch.zeros_like(avg),
                "lib": gpu.load_library()}
    dim, n = case["dim"], case["blocks"]
    order = list(range(n))
    random.Random(seed).shuffle(order)
    avg = _haloed(dim, n, seed)
    surfaces = torch.zeros((n, 6, dim + 2, IC, IC if dim == 3 else 1), dtype=torch.float64, device=DEV)
    ti = lts.LevelTimeIntegrator(dim)
    for dt in (1.0e-4, 1.1e-4):
        ti.append_micro_timestep(dt)
    lib, ctx = gpu.load_library(), ctypes.c_void_p()
    gpu.check(lib.alpaca_context_create(gpu._stream_ptr(), ctypes.byref(ctx)), "context_create")
    side = max(1, int(round(n ** (1.0 / dim))))
    nb = [side] * (dim - 1) + [n // side ** (dim - 1)]
    grid = nb[0] * nb[1] * (nb[2] if dim == 3 else 1)
    return {"kind": kind, "dim": dim, "n": n, "lib": lib, "ctx": ctx, "ti": ti,
            "desc": gpu.make_desc(dim, [n] + [1] * (dim - 1), [gpu.BC_ZERO_GRADIENT] * dim,
                                  flux=FLUX[case["flux"]], precision=FORM[case["form"]],
                                  cell_size=1.0 / 64),
            "list": torch.tensor(order, dtype=torch.int32, device=DEV), "avg": avg,
            "init": _haloed(dim, n, seed + 1), "rhs": torch.zeros_like(avg), "flux": surfaces,
            "cons": torch.zeros_like(surfaces), "new": torch.zeros_like(avg), "work": avg.clone(),
            "table": torch.from_numpy(gpu.grid_neighbors(dim, nb, [gpu.BC_PERIODIC] * dim)).to(DEV),
            "grid": grid}


# --------------------------------------------------------------------- runs

def run(state):
    kind = state["kind"]
    if kind == "uniform":
        state["case"].advance(state["steps"])
        return {"u": state["case"].u}
    if kind == "serve":
        ens = state["ens"]
        ids = [ens.add_case(d, u, 1e300, CFL, sync=False) for d, u in state["cases"]]
        for _ in range(state["steps"] // 8):  # a serving loop looks at the records every few steps
            ens.step(8)
            records = ens.states()
        out = {"%02d" % i: ens.case_blocks(c) for i, c in enumerate(ids)}
        out["steps"] = torch.tensor([records[c].steps for c in ids])
        for c in ids:
            ens.remove_case(c)
        return out
    if kind == "multilevel":
        sol = state["sol"]
        sol.advance()
        return {"nodes": sol.be.avg, "time": sol.current_run_time}
    if kind == "mr":
        b, dim, op = state["blocks"], state["dim"], state["op"]
        op.average(b, dim, state["links"])
        details, decisions = op.child_needs_remeshing(b, dim, state["links"])
        op.prediction(b, dim, state["fine"], (HS, IC) * dim)
        op.jump_halo_update(b, dim, state["jumps"], state["where"])
        return {"blocks": b, "decisions": decisions, "details": details}
    if kind == "rhs":
        gpu.check(state["lib"].alpaca_right_hand_side(
            ctypes.byref(state["desc"]), state["n"], _ptr(state["avg"]), _ptr(state["rhs"]),
            gpu._stream_ptr()), "right_hand_side")
        return {"rhs": state["rhs"]}
    lib, ti, dim, n, blocks = state["lib"], state["ti"], state["dim"], state["n"], state["list"]
    # One middle stage of a level: the same start each time (a copy that the first
    # stage's FillInitialBuffer makes), then the stage's operations.
    ti.fill_initial_buffer(state["avg"], state["work"], blocks, 0)
    gpu.check(lib.alpaca_ctx_right_hand_side_jump_fluxes_list(
        state["ctx"], ctypes.byref(state["desc"]), n, _ptr(blocks), n, _ptr(state["work"]),
        _ptr(state["rhs"]), _ptr(state["flux"])), "rhs_list")
    ti.prepare_buffer_for_integration(state["work"], state["init"], blocks, 1)
    ti.integrate_node(state["work"], state["rhs"], state["cons"], state["flux"], blocks, 1, 2)
    gpu.fill_halos_table(state["rhs"], dim, state["table"], [gpu.BC_PERIODIC] * (2 * dim))
    lts.reset_jump_conservatives(dim, state["cons"], blocks)
    return {"new": state["rhs"], "work": state["work"]}


# --------------------------------------------------------------------- work

def work(case):
    kind = case["kind"]
    d8 = 8.0
    if kind == "uniform":
        cells = IC ** case["dim"] * case["nx"] * case["ny"] * case["nz"]
        # Per step: stage 1 reads u and writes u1, stages 2 and 3 read two states and write one.
        return {"bytes": case["steps"] * cells * (case["dim"] + 2) * d8 * 8,
                "flops": case["steps"] * cells * 3 * FLOP_STAGE[case["dim"], case["flux"]]}
    if kind == "serve":
        cells = sum(s["nx"] * s["ny"] for s in _serve_specs(case, 0)) * IC * IC
        return {"bytes": cells * 4 * d8 * (8 * case["steps"] + 4),
                "flops": case["steps"] * cells * 3 * FLOP_STAGE[2, case["flux"]]}
    if kind == "multilevel":
        dim, lmax = case["dim"], case["lmax"]
        # About a third of the finest level's micro steps' cells are leaves' (the rest are coarse).
        cells = 0.33 * (case["n0"] * IC << lmax) ** dim * (1 << lmax)
        return {"bytes": cells * (dim + 2) * d8 * 8, "flops": cells * 3 * FLOP_STAGE[dim, case["flux"]]}
    if kind == "mr":
        dim = case["dim"]
        rows, fine, jumps, _ = _mr_rows(case)
        ne, links = dim + 2, len(rows)
        average = links * ne * (IC ** dim + (IC // 2) ** dim)
        details = links * 2 * (IC ** dim + TC ** dim)
        predict = len(fine) * ne * (IC ** dim + 12 ** dim)
        halo = len(jumps) * ne * 2 * HS * IC ** (dim - 1) / (1.0 if dim == 2 else 4.0)
        points = links * 2 * 12 ** dim + len(fine) * ne * 8 ** dim
        return {"bytes": d8 * (average + details + predict + halo),
                "flops": points * (600.0 if dim == 3 else 60.0)}
    dim, n = case["dim"], case["blocks"]
    block = (dim + 2) * TC ** dim * d8
    flops = n * IC ** dim * FLOP_STAGE[dim, case["flux"]]
    if kind == "rhs":
        return {"bytes": 2 * n * block, "flops": flops}
    return {"bytes": n * block * (2 + 2 + 3 + 3 + 1.5), "flops": flops}


# -------------------------------------------------------- 64-bit comparison
# The scheme in plain torch, from its mathematics: WENO5-JS on characteristic
# variables of the Roe average, HLLC with Einfeldt speeds or Roe flux splitting,
# SSP-RK3.

def _pressure(u, gamma, b):
    return (gamma - 1.0) * (u[1] - 0.5 * (u[2:] ** 2).sum(0) / u[0]) - gamma * b


def _weno(v1, v2, v3, v4, v5):
    eps = 1.0e-6
    s1 = 13.0 / 12.0 * (v1 - 2 * v2 + v3) ** 2 + 0.25 * (v1 - 4 * v2 + 3 * v3) ** 2
    s2 = 13.0 / 12.0 * (v2 - 2 * v3 + v4) ** 2 + 0.25 * (v2 - v4) ** 2
    s3 = 13.0 / 12.0 * (v3 - 2 * v4 + v5) ** 2 + 0.25 * (3 * v3 - 4 * v4 + v5) ** 2
    a1, a2, a3 = 0.1 / (s1 + eps) ** 2, 0.6 / (s2 + eps) ** 2, 0.3 / (s3 + eps) ** 2
    num = (a1 * (2 * v1 - 7 * v2 + 11 * v3) + a2 * (-v2 + 5 * v3 + 2 * v4) +
           a3 * (2 * v3 + 5 * v4 - v5))
    return num / (6.0 * (a1 + a2 + a3))


def _physical_flux(u, d, gamma, b):
    p = _pressure(u, gamma, b)
    vn = u[2 + d] / u[0]
    f = u * vn
    f[1] += p * vn
    f[2 + d] += p
    return f


def _face_flux(cell, d, flux, gamma, b):
    """Flux through the faces between cell[2] and cell[3] (six tensors [NE][...])
    along axis d; zero where the reconstruction is not admissible."""
    dim = cell[0].shape[0] - 2
    left, right = cell[2], cell[3]
    pl, pr = _pressure(left, gamma, b), _pressure(right, gamma, b)
    sl, sr = left[0].sqrt(), right[0].sqrt()
    mean = lambda x, y: (x * sl + y * sr) / (sl + sr)  # noqa: E731
    vl, vr = left[2:] / left[0], right[2:] / right[0]
    v = mean(vl, vr)
    h = mean((left[1] + pl) / left[0], (right[1] + pr) / right[0])
    psi = mean((pl + gamma * b) / left[0], (pr + gamma * b) / right[0])
    g = gamma - 1.0
    pod = mean(pl / left[0], pr / right[0]) + 0.5 * sl * sr / (sl + sr) ** 2 * ((vl - vr) ** 2).sum(0)
    cc = psi + g * pod
    c = cc.sqrt()
    q2 = (v * v).sum(0)
    vn, roe_rho = v[d], sl * sr
    others = [a for a in range(dim) if a != d]

    def project(x):
        """Amplitudes of the waves u-c, shear (one per other axis), entropy, u+c."""
        vm = (v * x[2:]).sum(0)
        acoustic = g * (q2 * x[0] - h * x[0] - vm + x[1])
        drift = vn * x[0] - x[2 + d]
        w = [0.5 / cc * (acoustic + cc * x[0] + c * drift)]
        w += [(x[2 + a] - v[a] * x[0]) / roe_rho for a in others]
        w.append(((h - q2) * x[0] + vm - x[1]) / cc)
        w.append(0.5 / cc * (acoustic + cc * x[0] - c * drift))
        return w

    def physical(w):
        out = torch.empty_like(cell[0])
        entropy = w[dim] * g
        out[0] = w[0] + entropy + w[dim + 1]
        out[2 + d] = (vn - c) * w[0] + entropy * vn + (vn + c) * w[dim + 1]
        energy = (h - vn * c) * w[0] + (g * h - cc) * w[dim] + (h + vn * c) * w[dim + 1]
        for a, s in zip(others, [x * roe_rho for x in w[1:dim]]):
            out[2 + a] = v[a] * (w[0] + entropy + w[dim + 1]) + s
            energy = energy + v[a] * s
        out[1] = energy
        return out

    if flux == "roe":
        speed = [(vn - c).abs()] + [vn.abs()] * dim + [(vn + c).abs()]
        waves = [project(x) for x in cell]
        fluxes = [project(_physical_flux(x, d, gamma, b)) for x in cell]
        total = []
        for k in range(dim + 2):
            up = [f[k] + speed[k] * w[k] for f, w in zip(fluxes, waves)]
            down = [f[k] - speed[k] * w[k] for f, w in zip(fluxes, waves)]
            total.append(0.5 * (_weno(*up[:5]) + _weno(*down[:0:-1])))
        return physical(total)

    waves = [project(x) for x in cell]
    cols = [[w[k] for w in waves] for k in range(dim + 2)]
    ul = physical([_weno(*x[:5]) for x in cols])
    ur = physical([_weno(*x[:0:-1]) for x in cols])
    del waves, cols
    pl, pr = _pressure(ul, gamma, b), _pressure(ur, gamma, b)
    ok = (ul[0] > 2.3e-16) & (ur[0] > 2.3e-16) & (pl > -b) & (pr > -b)
    wl, wr = ul[2 + d] / ul[0], ur[2 + d] / ur[0]
    al, ar = (gamma * (pl + b) / ul[0]).sqrt(), (gamma * (pr + b) / ur[0]).sqrt()
    sl, sr = ul[0].sqrt(), ur[0].sqrt()
    un = (wl * sl + wr * sr) / (sl + sr)
    ce = ((al * al * sl + ar * ar * sr) / (sl + sr) +
          0.5 * sl * sr / (sl + sr) ** 2 * (wr - wl) ** 2).sqrt()
    lo, hi = torch.minimum(un - ce, wl - al), torch.maximum(un + ce, wr + ar)
    ml, mrr = ul[0] * (lo - wl), ur[0] * (hi - wr)
    star = (pr - pl + wl * ml - wr * mrr) / (ml - mrr)

    def side(u, p, w, s, clamped):
        chi = (s - w) / (s - star)
        q = torch.empty_like(u)
        q[0] = u[0] * chi
        q[2 + d] = u[0] * chi * star
        q[1] = u[0] * chi * (u[1] / u[0] + (star - w) * (star + p / (u[0] * (clamped - w))))
        for a in others:
            q[2 + a] = chi * u[2 + a]
        return _physical_flux(u, d, gamma, b) + clamped * (q - u)

    fl = side(ul, pl, wl, lo, lo.clamp(max=0.0))
    fr = side(ur, pr, wr, hi, hi.clamp(min=0.0))
    sign = torch.sign(star)
    f = 0.5 * (1.0 + sign) * fl + 0.5 * (1.0 - sign) * fr
    return torch.where(ok, f, torch.zeros_like(f))


def _pad(u, d, kind, width):
    """u [NE][...] with `width` more cells at both ends of axis d (axis 1 + d)."""
    a, n = 1 + d, u.shape[1 + d]
    if kind == "p":
        at = torch.arange(-width, n + width, device=u.device) % n
        return u.index_select(a, at)
    if kind == "z":
        return u.index_select(a, torch.arange(-width, n + width, device=u.device).clamp(0, n - 1))
    at = torch.arange(-width, n + width, device=u.device)
    out = u.index_select(a, torch.where(at < 0, -1 - at, torch.where(at >= n, 2 * n - 1 - at, at)))
    for s in ((0, width), (n + width, width)):
        out[2 + d].narrow(d, *s).neg_()
    return out


def _rate(u, case, dx):
    """du/dt of the whole domain."""
    dim, out = case["dim"], torch.zeros_like(u)
    for d in range(dim):
        w = _pad(u, d, case["bc"][d], 3)
        faces = w.shape[1 + d] - 5
        f = _face_flux([w.narrow(1 + d, m, faces) for m in range(6)], d, case["flux"], case["gamma"],
                       case["b"])
        out += (f.narrow(1 + d, 0, faces - 1) - f.narrow(1 + d, 1, faces - 1)) / dx
        del w, f
    return out


def _advance(u, case, steps):
    dim = case["dim"]
    u = u[..., 0] if dim == 2 else u
    dx = 1.0 / (case["nx"] * IC)
    for _ in range(steps):
        c = (case["gamma"] * (_pressure(u, case["gamma"], case["b"]) + case["b"]) / u[0]).sqrt()
        dt = CFL * dx / ((u[2:] / u[0]).abs().sum(0) + dim * c).max()
        u1 = u + dt * _rate(u, case, dx)
        u2 = 0.75 * u + 0.25 * (u1 + dt * _rate(u1, case, dx))
        u = (u + 2.0 * (u2 + dt * _rate(u2, case, dx))) / 3.0
    return u


def _to_blocks(u, case):
    """Haloed blocks of a domain state: the four halo layers of every block face,
    zero in edges and corners."""
    dim, nb = case["dim"], _nb(case)
    out = torch.zeros(nb + [dim + 2] + [TC] * dim, dtype=torch.float64, device=u.device)
    for d in range(dim):
        w = _pad(u, d, case["bc"][d], HS).unfold(1 + d, TC, IC)
        for a in range(dim):
            if a != d:
                w = w.unfold(1 + a, IC, IC)
        # unfold appends the window axes: d first, then the others in order.
        window = [1 + dim + ([d] + [a for a in range(dim) if a != d]).index(a) for a in range(dim)]
        w = w.permute(list(range(1, 1 + dim)) + [0] + window)
        out[(Ellipsis,) + tuple(slice(None) if a == d else slice(HS, HS + IC) for a in range(dim))] = w
    return out


def _blocks_rate(avg, dim, flux, dx, gamma=1.4, b=0.0):
    """Right-hand side of haloed blocks [n][NE][24]...: internal cells, zero halos."""
    u = avg.reshape(avg.shape[:2] + (TC,) * dim).transpose(0, 1)
    inner = u
    for a in range(dim):
        inner = inner.narrow(2 + a, HS, IC)
    total = torch.zeros_like(inner)
    for d in range(dim):
        w = u
        for a in range(dim):
            if a != d:
                w = w.narrow(2 + a, HS, IC)
        f = _face_flux([w.narrow(2 + d, HS - 3 + m, IC + 1) for m in range(6)], d, flux, gamma, b)
        total += (f.narrow(2 + d, 0, IC) - f.narrow(2 + d, 1, IC)) / dx
    out = torch.zeros_like(u)
    view = out
    for a in range(dim):
        view = view.narrow(2 + a, HS, IC)
    view.copy_(total)
    return out.transpose(0, 1).reshape(avg.shape).contiguous()


def _predict(parent, position, dim):
    """The child's whole block from its parent [NE][24].. (a tensor product of the
    one-dimensional fifth-order prediction)."""
    out = parent
    for a in range(dim):
        first = 10 if (position >> a) & 1 else 2
        at = lambda k: out.narrow(1 + a, first + k, 12)  # noqa: B023,E731
        slope = -22.0 / 128.0 * (at(1) - at(-1)) + 3.0 / 128.0 * (at(2) - at(-2))
        pair = torch.stack([at(0) + slope, at(0) - slope], dim=2 + a)
        out = pair.flatten(1 + a, 2 + a)
    return out


def _exact_mr(case, seed):
    dim = case["dim"]
    rows, fine, jumps, n = _mr_rows(case)
    if len(rows) + len(jumps) > 9000:
        return None
    b = _haloed(dim, n, seed)
    b = b.reshape(b.shape[:2] + (TC,) * dim)
    parent = torch.tensor([r[1] for r in rows], device=DEV)
    position = [r[2] for r in rows]
    for child, par, pos, _ in rows:
        c = b[child]
        for a in range(dim):
            c = c.narrow(1 + a, HS, IC).unflatten(1 + a, (IC // 2, 2)).mean(2 + a)
        half = [TC // 2 if (pos >> a) & 1 else HS for a in range(dim)]
        b[(par, slice(None)) + tuple(slice(h, h + IC // 2) for h in half)] = c
    details = torch.stack([((b[r[0]][:2] - _predict(b[r[1]], r[2], dim)[:2]).abs() /
                            b[r[0]][:2].abs()).max() for r in rows])
    del parent, position
    inner = (slice(None),) + (slice(HS, HS + IC),) * dim
    for child, par, pos, _ in fine:
        b[child][inner] = _predict(b[par], pos, dim)[inner]
    for (child, par, pos, _), loc in jumps:
        r = mr.halo_recv_range(dim, loc)
        at = (slice(None),) + tuple(slice(r[2 * a], r[2 * a] + r[2 * a + 1]) for a in range(dim))
        b[child][at] = _predict(b[par], pos, dim)[at]
    return {"blocks": b if dim == 3 else b[..., None], "decisions": None, "details": details}


def exact(case, seed):
    kind = case["kind"]
    if kind == "uniform":
        u = _field(case["dim"], [m * IC for m in _nb(case)], seed, case["gamma"], case["b"])
        u = _to_blocks(_advance(u, case, case["steps"]), case)
        ne, dim = case["dim"] + 2, case["dim"]
        return {"u": u.reshape((-1, ne) + (TC,) * dim)}
    if kind == "serve":
        out = {"steps": None}
        for i, s in enumerate(_serve_specs(case, seed)):
            u = _field(2, [s["nx"] * IC, s["ny"] * IC], s["seed"], s["gamma"], 0.0)
            out["%02d" % i] = _to_blocks(_advance(u, s, case["steps"]), s).reshape(-1)
        return out
    if kind == "mr":
        return _exact_mr(case, seed)
    if kind == "rhs":
        return {"rhs": _blocks_rate(_haloed(case["dim"], case["blocks"], seed), case["dim"],
                                    case["flux"], 1.0 / 64)}
    return None  # multilevel: the whole driver; level: its pieces are held by the other kinds
