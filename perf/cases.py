"""The work that users of this package run on the GPU, as measurable cases.

Every case goes through the package's public entry points: the device-resident
Simulation (step loops and evolve), the reverse mode, self-gravity, block meshes
with and without dynamic refinement, the ghosted MUSCL grid, and the per-face flux
backend on host arrays. `listed()` names twelve of them, `draw()` gives more of the
same ranges. `exact()` restates the arithmetic in Float64 torch, independent of the
package.
"""
import ctypes
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.getcwd()


def _package():
    """vespa.jl_amd/ holds a dot in its name: it is loaded as `vespa_jl_amd`."""
    if "vespa_jl_amd" not in sys.modules:
        d = os.path.join(ROOT, "vespa.jl_amd")
        spec = importlib.util.spec_from_file_location("vespa_jl_amd", os.path.join(d, "__init__.py"),
                                                      submodule_search_locations=[d])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["vespa_jl_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["vespa_jl_amd"]


# ------------------------------------------------------------------ the cases


def listed():
    return [
        # The benchmark's headline run: a periodic turbulence box, fast arithmetic.
        {"name": "box 256^3 f64", "kind": "grid", "rank": 3, "nx": 256, "ny": 256, "nz": 256, "bc": "periodic",
         "f32": False, "mode": "fast", "evolve": False, "steps": 2},
        # A 3D flow between walls on a ragged grid, Float32, the default arithmetic, run by evolve().
        {"name": "channel 171x130x97 f32", "kind": "grid", "rank": 3, "nx": 171, "ny": 130, "nz": 97, "bc": "walls",
         "f32": True, "mode": "exact", "evolve": True, "steps": 4},
        # A 2D shear layer at the resolution of the reverse-mode benchmark, run by evolve().
        {"name": "layer 512^2 f64", "kind": "grid", "rank": 2, "nx": 512, "ny": 512, "nz": 1, "bc": "periodic",
         "f32": False, "mode": "exact", "evolve": True, "steps": 20},
        # The shock tube of the tests and the benchmark: 400 cells to t = 0.2, all latency.
        {"name": "tube 400 f64", "kind": "tube", "nx": 400, "bc": "outflow", "f32": False, "mode": "exact"},
        # Gradient of a 2D rollout with respect to its initial state, checkpoints every 20 steps.
        {"name": "gradient 512^2 x 60", "kind": "rollout", "nx": 512, "ny": 512, "steps": 60, "every": 20},
        # Pullback of one step on a small bounded 3D grid (the general reverse-mode form), host arrays.
        {"name": "pullback 60x52x44", "kind": "vjp", "rank": 3, "nx": 60, "ny": 52, "nz": 44, "bc": "walls"},
        # Self-gravitating gas in a periodic box: a Poisson solve and a sourced step, by evolve().
        {"name": "gravity 128^3 f64", "kind": "gravity", "nx": 128, "ny": 128, "nz": 128, "bc": "periodic",
         "f32": False, "steps": 1},
        # Batched uneven blocks, conforming and 2:1 links, an output every 50 steps.
        {"name": "blocks 400 f64", "kind": "blocks", "blocks": 400, "f32": False, "mode": "fast", "steps": 50},
        # Blast wave with dynamic refinement, the whole run with its regrids.
        {"name": "blast amr f64", "kind": "amr", "nroot": 6, "maxlevel": 3, "tfinal": 0.02, "f32": False},
        # The published MUSCL workload: 256^3 cells and 4 ghost zones, Float32, a periodic box.
        {"name": "muscl 256^3 f32", "kind": "muscl", "nx": 256, "ny": 256, "nz": 256, "ng": 4, "f32": True,
         "mode": "exact", "dual": False, "record": False, "bc": True, "steps": 2},
        # One subgrid of a refined hierarchy: ghosts set by its parent, dual energy, fluxes recorded for the reflux.
        {"name": "muscl subgrid 42x36x30 f64", "kind": "muscl", "nx": 42, "ny": 36, "nz": 30, "ng": 3, "f32": False,
         "mode": "exact", "dual": True, "record": True, "bc": False, "steps": 1},
        # The flux backend on a batch of host face states, as a solver's gather pass hands them over.
        {"name": "faces 200000 f64", "kind": "faces", "faces": 200000, "f32": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["grid", "grid", "grid", "tube", "rollout", "vjp", "gravity", "blocks", "amr", "muscl", "muscl",
                       "faces"])
    f32 = rng.random() < 0.4
    mode = rng.choice(["exact", "fast"])
    if kind == "grid":
        rank = rng.choice([2, 3, 3])
        n = [_log_int(rng, 24, 230) for _ in range(3)] if rank == 3 else [_log_int(rng, 40, 1400) for _ in range(2)] + [1]
        return {"kind": kind, "rank": rank, "nx": n[0], "ny": n[1], "nz": n[2],
                "bc": rng.choice(["periodic", "walls", "outflow"]), "f32": f32, "mode": mode,
                "evolve": rng.random() < 0.6, "steps": rng.randint(2, 8)}
    if kind == "tube":
        return {"kind": kind, "nx": _log_int(rng, 60, 2000), "bc": rng.choice(["outflow", "reflecting"]), "f32": f32,
                "mode": mode}
    if kind == "rollout":
        return {"kind": kind, "nx": 32 * rng.randint(2, 16), "ny": 16 * rng.randint(4, 32),
                "steps": rng.randint(10, 60), "every": rng.choice([5, 10, 20])}
    if kind == "vjp":
        rank = rng.choice([2, 3])
        n = [_log_int(rng, 16, 72) for _ in range(3)] if rank == 3 else [_log_int(rng, 40, 500) for _ in range(2)] + [1]
        return {"kind": kind, "rank": rank, "nx": n[0], "ny": n[1], "nz": n[2], "bc": rng.choice(["periodic", "walls"])}
    if kind == "gravity":
        n = [_log_int(rng, 20, 128) for _ in range(3)]
        return {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2], "bc": rng.choice(["periodic", "walls"]), "f32": f32,
                "steps": rng.randint(1, 2)}
    if kind == "blocks":
        return {"kind": kind, "blocks": _log_int(rng, 40, 400), "f32": f32, "mode": mode, "steps": rng.randint(20, 50)}
    if kind == "amr":
        return {"kind": kind, "nroot": rng.randint(4, 8), "maxlevel": rng.randint(1, 3),
                "tfinal": round(rng.uniform(0.004, 0.02), 4), "f32": f32}
    if kind == "muscl":
        n = [_log_int(rng, 16, 200) for _ in range(3)]
        dual, record = rng.random() < 0.4, max(n) < 64 and rng.random() < 0.6
        return {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2], "ng": rng.randint(2, 4), "f32": f32, "mode": mode,
                "dual": dual, "record": record, "bc": rng.random() < 0.6, "steps": 1 if record else rng.randint(1, 4)}
    return {"kind": "faces", "faces": _log_int(rng, 500, 400000), "f32": f32}


# ------------------------------------------------------------------ inputs


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(1000003 + int(seed))


def _modes(dims, seed, fields, kmax=4, nmodes=6):
    """(fields, [nz,] [ny,] nx) Float64: random-phase cosines of integer wave
    vectors, about unit RMS each."""
    rng = np.random.default_rng(seed)
    rank = len(dims)
    x = [(torch.arange(n, dtype=torch.float64, device="cuda") + 0.5) / n for n in dims]
    out = torch.zeros((fields,) + tuple(reversed(dims)), dtype=torch.float64, device="cuda")
    for f in range(fields):
        for _ in range(nmodes):
            k = rng.integers(-kmax, kmax + 1, rank)
            ph = torch.full((), float(rng.uniform(0, 2 * np.pi)), dtype=torch.float64, device="cuda")
            for d in range(rank):
                ph = ph + (2 * np.pi * int(k[d]) * x[d]).reshape([-1 if e == d else 1 for e in reversed(range(rank))])
            out[f] += math.sqrt(2.0 / nmodes) * torch.cos(ph)
    return out


def _cons(W, gamma):
    r, vx, vy, vz, p = W
    return torch.stack([r, r * vx, r * vy, r * vz, p / (gamma - 1) + 0.5 * r * (vx * vx + vy * vy + vz * vz)])


GAMMA = 5.0 / 3.0


def _grid_state(c, seed):
    """A smooth subsonic flow; in 2D a perturbed shear layer."""
    dims = [c["nx"], c["ny"], c["nz"]][:c["rank"]]
    m = _modes(dims, seed, 5)
    r = 1.0 + 0.1 * m[0]
    v = [0.12 * m[1], 0.12 * m[2], 0.12 * m[3]]
    p = 1.0 + 0.05 * m[4]
    if c["rank"] == 2:
        y = ((torch.arange(dims[1], dtype=torch.float64, device="cuda") + 0.5) / dims[1]).reshape(-1, 1)
        prof = 0.5 * (torch.tanh((y - 0.25) / 0.05) - torch.tanh((y - 0.75) / 0.05))
        r = r + 0.5 * prof
        v[0] = 0.1 * m[1] + (prof - 0.5)
        v[2] = torch.zeros_like(r)
        p = p + 1.5
    return _cons(torch.stack([r, v[0], v[1], v[2], p]), GAMMA)


def _codes(c):
    """Boundary conditions per axis (lo, hi): walls are reflecting across x, outflow
    along y, periodic along z."""
    rank = c.get("rank", 3)
    if c["bc"] == "periodic":
        return [("periodic", "periodic")] * rank
    if c["bc"] == "outflow":
        return [("outflow", "outflow")] * rank
    return [("reflecting", "reflecting"), ("outflow", "outflow"), ("periodic", "periodic")][:rank]


def _simulation(V, dims, bcs, f32, mode, tfinal=1e9, cfl=0.3):
    prob = V.Problem("case", tuple(dims), ((0.0, 1.0),) * len(dims), GAMMA, bcs,
                     lambda x, y, z: (1.0, 0.0, 0.0, 0.0, 1.0), tfinal, cfl)
    sim = V.Simulation(V.UniformMesh(tuple(dims), prob.domain), prob, eltype=np.float32 if f32 else np.float64)
    sim.set_mode(mode)
    return sim


class _Device:
    """A device pointer of the library, for torch."""

    def __init__(self, ptr, shape, f32):
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4" if f32 else "<f8",
                                         "data": (int(ptr), False), "version": 2, "strides": None}


def _view(owner, ptr, shape, f32):
    """The memory as a tensor (no copy) that keeps alive the object that owns it."""
    t = torch.as_tensor(_Device(ptr, shape, f32), device="cuda")
    t.owner = owner
    return t


def _fill(view, U):
    view.copy_(U)
    torch.cuda.synchronize()


def _tube_state(c, seed):
    rng = np.random.default_rng(seed)
    n = c["nx"]
    x = (np.arange(n) + 0.5) / n
    left = x < rng.uniform(0.45, 0.55)
    W = np.zeros((5, n))
    W[0] = np.where(left, rng.uniform(0.9, 1.1), rng.uniform(0.1, 0.15))
    W[4] = np.where(left, rng.uniform(0.9, 1.1), rng.uniform(0.09, 0.11))
    return np.stack([W[0], W[1], W[2], W[3], W[4] / (GAMMA - 1)])


def _gravity_state(c, seed):
    dims = [c["nx"], c["ny"], c["nz"]]
    r = 1.0 + 0.05 * _modes(dims, seed, 1, kmax=3)[0]
    r = r + 1e-3 * torch.randn(r.shape, dtype=torch.float64, device="cuda", generator=_gen(seed))
    z = torch.zeros_like(r)
    return _cons(torch.stack([r, z, z, z, 1.0 + z]), GAMMA)


def _muscl_state(c, seed):
    """The turbulence state of the MUSCL benchmark in kind: ρ near 1, c_s near 1,
    RMS Mach 0.3, with the gas energy as the sixth field under dual energy."""
    dims = [c["nx"] + 2 * c["ng"], c["ny"] + 2 * c["ng"], c["nz"] + 2 * c["ng"]]
    m = _modes(dims, seed, 5, kmax=3)
    r = 1.0 + 0.05 * m[0]
    v = 0.17 * m[1:4]
    ge = (1.0 / 1.4) / 0.4 * (1.0 + 0.05 * m[4])
    U = [r, r * v[0], r * v[1], r * v[2], r * (ge + 0.5 * (v * v).sum(0))]
    if c["dual"]:
        U.append(r * ge)
    return torch.stack(U)


def _muscl_dims(c):
    return (c["nx"] + 2 * c["ng"], c["ny"] + 2 * c["ng"], c["nz"] + 2 * c["ng"])


def _muscl_dt(c):
    return 0.2 / max(c["nx"], c["ny"], c["nz"])


def _face_states(c, seed):
    rng = np.random.default_rng(seed)
    n, T = c["faces"], np.float32 if c["f32"] else np.float64
    WL = np.empty((n, 5))
    WL[:, 0], WL[:, 1:4], WL[:, 4] = rng.uniform(0.2, 3, n), rng.uniform(-1.5, 1.5, (n, 3)), rng.uniform(0.1, 3, n)
    WR = WL * (1 + 0.2 * rng.uniform(-1, 1, (n, 5)))
    return WL.astype(T), WR.astype(T), rng.integers(1, 4, n).astype(np.int32)


def prepare(c, seed):
    V = _package()
    kind = c["kind"]
    T = np.float32 if c.get("f32") else np.float64
    if kind == "grid":
        dims = [c["nx"], c["ny"], c["nz"]][:c["rank"]]
        sim = _simulation(V, dims, _codes(c), c["f32"], c["mode"])
        view = _view(sim, sim.device_state_ptr(), sim.shape, c["f32"])
        _fill(view, _grid_state(c, seed))
        return {"kind": kind, "sim": sim, "view": view, "evolve": c["evolve"], "steps": c["steps"]}
    if kind == "tube":
        sim = _simulation(V, [c["nx"]], c["bc"], c["f32"], c["mode"], tfinal=0.2, cfl=0.4)
        return {"kind": kind, "sim": sim, "U0": _tube_state(c, seed).astype(T)}
    if kind == "rollout":
        from vespa_jl_amd import adjoint
        sim = _simulation(V, [c["nx"], c["ny"]], "periodic", False, "exact", cfl=0.4)
        U0 = _grid_state(dict(c, rank=2, nz=1), seed).cpu().numpy()
        w = torch.randn(sim.shape, dtype=torch.float64, device="cuda", generator=_gen(seed)).cpu().numpy()
        return {"kind": kind, "sim": sim, "U0": U0, "w": w, "ro": adjoint.Rollout(sim, c["steps"], c["every"])}
    if kind == "vjp":
        dims = [c["nx"], c["ny"], c["nz"]][:c["rank"]]
        sim = _simulation(V, dims, _codes(c), False, "exact")
        U = _grid_state(c, seed).cpu().numpy()
        w = torch.randn(sim.shape, dtype=torch.float64, device="cuda", generator=_gen(seed)).cpu().numpy()
        return {"kind": kind, "sim": sim, "U": U, "w": w, "dt": 0.1 / max(dims)}
    if kind == "gravity":
        sim = _simulation(V, [c["nx"], c["ny"], c["nz"]], _codes(c), c["f32"], "exact")
        view = _view(sim, sim.device_state_ptr(), sim.shape, c["f32"])
        _fill(view, _gravity_state(c, seed))
        grav = V.enable_gravity(sim, G=1.0, bcs="periodic" if c["bc"] == "periodic" else "neumann",
                                project_mean=True)
        return {"kind": kind, "sim": sim, "view": view, "grav": grav, "steps": c["steps"]}
    if kind == "blocks":
        from vespa_jl_amd import blockmesh
        mesh = blockmesh.random_block_pairs(c["blocks"], seed=c["blocks"], rank=3)   # one layout per size
        sim = blockmesh.BlockSimulation(mesh, T, cfl=0.3)
        sim.set_mode(c["mode"])
        sim.upload(blockmesh.smooth_block_state(mesh, seed, dtype=T))
        return {"kind": kind, "sim": sim, "steps": c["steps"]}
    if kind == "amr":
        from vespa_jl_amd import amr
        qb = amr.QuadBlocks(c["nroot"], 8, c["maxlevel"])
        U0 = amr.sedov_quadblocks_state(qb, r_hot=0.05)
        U0[0] *= 1.0 + 1e-3 * np.random.default_rng(seed).uniform(-1, 1, U0.shape[1])
        return {"kind": kind, "U0": U0.astype(T), "nroot": c["nroot"], "maxlevel": c["maxlevel"],
                "tfinal": c["tfinal"], "T": T}
    if kind == "muscl":
        g = V.MusclGrid(_muscl_dims(c), c["ng"], 1.4, 1.5, 1.0 / max(c["nx"], c["ny"], c["nz"]), eltype=T,
                        dual=c["dual"])
        g.set_mode(c["mode"])
        if c["bc"]:
            g.set_bc("periodic")
        p = ctypes.c_void_p()
        V.check(V.load_library().vh_muscl_state_device_ptr(g._h, ctypes.byref(p)))
        view = _view(g, p.value, (g.nf,) + _muscl_dims(c)[::-1], c["f32"])
        _fill(view, _muscl_state(c, seed))
        return {"kind": kind, "grid": g, "view": view, "record": c["record"], "steps": c["steps"], "dt": _muscl_dt(c)}
    WL, WR, axis = _face_states(c, seed)
    return {"kind": kind, "backend": V.HIPFlux(), "model": V.IdealHydro(GAMMA), "WL": WL, "WR": WR, "axis": axis,
            "F": np.empty_like(WL)}


# ------------------------------------------------------------------ one pass


def run(s):
    V = _package()
    kind = s["kind"]
    if kind == "grid":
        if s["evolve"]:
            V.evolve(s["sim"], max_steps=s["steps"])
        else:
            V.run_steps(s["sim"], s["steps"])
        return s["view"]
    if kind == "tube":
        sim = s["sim"]
        sim.upload(s["U0"])
        sim.t, sim.step_count = 0.0, 0
        V.evolve(sim)
        return sim.state()
    if kind == "rollout":
        s["sim"].upload(s["U0"])
        UF = s["ro"].forward()
        return {"final": UF, "gradient": s["ro"].backward(s["w"])}
    if kind == "vjp":
        from vespa_jl_amd import adjoint
        return adjoint.step_vjp(s["sim"], s["U"], s["dt"], s["w"])
    if kind == "gravity":
        V.evolve(s["sim"], max_steps=s["steps"])
        return {"state": s["view"], "phi": s["grav"].phi()}
    if kind == "blocks":
        s["sim"].evolve(max_steps=s["steps"])
        return s["sim"].state()
    if kind == "amr":
        from vespa_jl_amd import amr
        qb = amr.QuadBlocks(s["nroot"], 8, s["maxlevel"])
        r = amr.evolve_amr(qb, s["U0"], s["tfinal"], cfl=0.4, dtype=s["T"])
        return {"U": r["U"], "t": r["t"], "steps": r["steps"], "leaves": r["leaves"]}
    if kind == "muscl":
        from vespa_jl_amd import muscl
        for _ in range(s["steps"]):
            s["grid"].step(s["dt"], fluxrec=s["record"])
        if not s["record"]:
            return s["view"]
        return {"state": s["view"], "fluxes": [list(a) for a in muscl.flux_register_arrays(s["grid"], s["dt"])]}
    return V.compute_face_fluxes(s["backend"], s["model"], s["F"], s["WL"], s["WR"], s["axis"])


# ------------------------------------------------------------------ the work a pass cannot do without


def work(c):
    """Bytes: each state read and written once per RK stage as SSP-RK2 needs it (stage
    1 reads and writes it, stage 2 reads both and writes one: 5 passes); flops: about
    100 per face flux, 20 per slope set and field sweep."""
    kind, e = c["kind"], 4 if c.get("f32") else 8
    cells = c.get("nx", 1) * c.get("ny", 1) * c.get("nz", 1)
    if kind == "grid":
        return {"bytes": 25 * e * cells * c["steps"], "flops": 2 * 150 * c["rank"] * cells * c["steps"]}
    if kind == "tube":
        return {"bytes": 10 * e * cells, "flops": 2 * 150 * cells * 1.1 * c["nx"]}
    if kind == "rollout":
        return {"bytes": 25 * e * cells * c["steps"] + 60 * e * cells * c["steps"],
                "flops": (600 + 1800) * cells * c["steps"]}
    if kind == "vjp":
        return {"bytes": 15 * e * cells, "flops": (150 + 900) * c["rank"] * cells}
    if kind == "gravity":
        return {"bytes": (25 + 2) * e * cells * c["steps"], "flops": 900 * cells * c["steps"]}
    if kind == "blocks":
        cells = 12500 * c["blocks"]
        return {"bytes": 25 * e * cells * c["steps"], "flops": 900 * cells * c["steps"]}
    if kind == "amr":
        cells = 64 * c["nroot"] ** 2 * 4
        steps = 6000 * c["tfinal"]
        return {"bytes": 25 * e * cells * steps, "flops": 600 * cells * steps}
    if kind == "muscl":
        nf = 6 if c["dual"] else 5
        n = _muscl_dims(c)
        cells = n[0] * n[1] * n[2]
        extra = 3 * nf * e + 15 * 8 if c["record"] else 0
        return {"bytes": (5 * nf * e + extra) * cells * c["steps"], "flops": 900 * cells * c["steps"]}
    return {"bytes": 15 * e * c["faces"], "flops": 100 * c["faces"]}


# ------------------------------------------------------------------ the same in Float64 torch


def _c2p(U, g):
    r = U[0]
    v = U[1:4] / r
    kin = 0.5 * r * (v * v).sum(0)
    p = (g - 1) * (U[4] - kin)
    return torch.cat([U[:1], v, torch.where(1e-12 * kin > p, 1e-12 * kin, p)[None]])


def _minmod(a, b):
    return torch.where(a * b <= 0, torch.zeros_like(a), torch.where(a.abs() < b.abs(), a, b))


def _ghost(W, bc, d):
    if bc != "reflecting":
        return W
    s = torch.ones((5,) + (1,) * (W.dim() - 1), dtype=W.dtype, device=W.device)
    s[1 + d] = -1
    return W * s


def _hllc(L, R, g, d):
    def energy(W):
        return W[4] / (g - 1) + 0.5 * W[0] * (W[1:4] * W[1:4]).sum(0)

    def flux(W):
        un = W[1 + d]
        m = [W[0] * W[1 + i] * un for i in range(3)]
        m[d] = m[d] + W[4]
        return torch.stack([W[0] * un, m[0], m[1], m[2], (energy(W) + W[4]) * un])

    def star(W, S, Ss):
        un, E = W[1 + d], energy(W)
        f = W[0] * (S - un) / (S - Ss)
        Us = torch.stack([f, f * (Ss if d == 0 else W[1]), f * (Ss if d == 1 else W[2]), f * (Ss if d == 2 else W[3]),
                          f * (E / W[0] + (Ss - un) * (Ss + W[4] / (W[0] * (S - un))))])
        return flux(W) + S * (Us - torch.stack([W[0], W[0] * W[1], W[0] * W[2], W[0] * W[3], E]))

    cL, cR = (g * L[4] / L[0]).sqrt(), (g * R[4] / R[0]).sqrt()
    uL, uR = L[1 + d], R[1 + d]
    SL = torch.where(uL - cL <= uR - cR, uL - cL, uR - cR)
    SR = torch.where(uL + cL >= uR + cR, uL + cL, uR + cR)
    Ss = (R[4] - L[4] + L[0] * uL * (SL - uL) - R[0] * uR * (SR - uR)) / (L[0] * (SL - uL) - R[0] * (SR - uR))
    F = torch.where(Ss >= 0, star(L, SL, Ss), star(R, SR, Ss))
    return torch.where(SL >= 0, flux(L), torch.where(SR <= 0, flux(R), F))


def _divergence(U, g, bcs, widths):
    """Sum over axes of (F_hi − F_lo)/w."""
    W = _c2p(U, g)
    out = torch.zeros_like(U)
    for d, (lo, hi) in enumerate(bcs):
        t = W.dim() - 1 - d
        n = W.shape[t]
        first, last = W.narrow(t, 0, 1), W.narrow(t, n - 1, 1)
        per = lo == "periodic"
        P = torch.cat([last if per else _ghost(first, lo, d), W, first if per else _ghost(last, hi, d)], t)
        s = _minmod(W - P.narrow(t, 0, n), P.narrow(t, 2, n) - W)
        a, b = W - 0.5 * s, W + 0.5 * s   # lo- and hi-face values
        a0, bn = a.narrow(t, 0, 1), b.narrow(t, n - 1, 1)
        L = torch.cat([bn if per else _ghost(a0, lo, d), b], t)
        R = torch.cat([a, a0 if per else _ghost(bn, hi, d)], t)
        F = _hllc(L, R, g, d)
        out = out + (F.narrow(t, 1, n) - F.narrow(t, 0, n)) / widths[d]
    return out


def _ref_dt(U, g, widths, cfl, rho_term=0.0):
    W = _c2p(U, g)
    c = (g * W[4] / W[0]).sqrt()
    m = max(float(((W[1 + d].abs() + c) / w).max()) for d, w in enumerate(widths))
    if rho_term:
        m = max(m, 2.0 * math.sqrt(rho_term * float(W[0].max())))
    return cfl / m


def _ref_step(U, dt, g, bcs, widths, source=None):
    def change(X):
        return _divergence(X, g, bcs, widths) + (source(X) if source else 0.0)
    U1 = U - dt * change(U)
    return 0.5 * U + 0.5 * (U1 - dt * change(U1))


def _poisson(rho, widths, periodic):
    """φ of ∇²φ = 4π(ρ − ρ̄) with the 7-point Laplacian, mean zero; Neumann sides
    through the even extension."""
    b = 4 * math.pi * (rho - rho.mean())
    if not periodic:
        for t in range(3):
            b = torch.cat([b, b.flip(t)], t)
    lam = torch.zeros_like(b)
    for d in range(3):
        n = b.shape[2 - d]
        k = torch.arange(n, dtype=torch.float64, device=b.device)
        lam = lam + ((2 * torch.cos(2 * math.pi * k / n) - 2) / widths[d] ** 2).reshape(
            [-1 if e == 2 - d else 1 for e in range(3)])
    lam[0, 0, 0] = 1.0
    f = torch.fft.fftn(b) / lam
    f[0, 0, 0] = 0
    phi = torch.fft.ifftn(f).real
    return phi[:rho.shape[0], :rho.shape[1], :rho.shape[2]].contiguous()


def _gravity_source(phi, widths, periodic):
    g = []
    for d in range(3):
        t = 2 - d
        n = phi.shape[t]
        lo, hi = torch.roll(phi, 1, t), torch.roll(phi, -1, t)
        dist = torch.full([n if e == t else 1 for e in range(3)], 2 * widths[d], dtype=torch.float64, device=phi.device)
        if not periodic:
            lo = torch.cat([phi.narrow(t, 0, 1), phi.narrow(t, 0, n - 1)], t)
            hi = torch.cat([phi.narrow(t, 1, n - 1), phi.narrow(t, n - 1, 1)], t)
            dist.narrow(t, 0, 1).fill_(1.5 * widths[d])
            dist.narrow(t, n - 1, 1).fill_(1.5 * widths[d])
        g.append(-(hi - lo) / dist)
    g = torch.stack(g)

    def source(U):
        return torch.cat([torch.zeros_like(U[:1]), -U[:1] * g, -(U[1:4] * g).sum(0)[None]])
    return source


def _ref_muscl_fluxes(U, c, dt):
    """HLL fluxes along each axis through the faces ng..n−ng, and dU."""
    g, th, small, ng, nf = 1.4, 1.5, 1e-10, c["ng"], U.shape[0]
    v = U[1:4] / U[0]
    v2 = (v * v).sum(0)
    e = U[4] / U[0] - 0.5 * v2
    if nf == 6:
        dual = U[5] / U[0]
        cs2 = torch.where(e > 0, g * (g - 1) * e, torch.zeros_like(e))
        e = torch.where((cs2 > 1e-3 * v2) & (e > 0.5 * dual), e, dual)
    W = torch.cat([U[:1], e.clamp_min(small)[None], v])
    dtdx = dt * max(c["nx"], c["ny"], c["nz"])
    dU, faces = torch.zeros_like(U), []
    for d in range(3):
        t = 3 - d
        n = W.shape[t]
        na = n - 2 * ng
        w = W.narrow(t, ng - 2, na + 4)
        m, x, p = w.narrow(t, 0, na + 2), w.narrow(t, 1, na + 2), w.narrow(t, 2, na + 2)
        a, b, q = (x - m) * th, (p - x) * th, 0.5 * (p - m)
        mn = torch.minimum(a.abs(), torch.minimum(b.abs(), q.abs()))
        s = torch.where((a > 0) & (b > 0) & (q > 0), mn, torch.where((a <= 0) & (b <= 0) & (q <= 0), -mn, 0 * mn))
        L, R = (x + 0.5 * s).narrow(t, 0, na + 1), (x - 0.5 * s).narrow(t, 1, na + 1)

        def side(S):
            r, ei, u = S[0].clamp_min(small), S[1], S[2 + d]
            et = ei + 0.5 * (S[2:5] * S[2:5]).sum(0)
            pr = (g - 1) * r * ei
            cs = (g * pr / r).sqrt()
            C = [r, r * S[2], r * S[3], r * S[4], r * et]
            F = [k * u for k in C]
            F[1 + d] = F[1 + d] + pr
            F[4] = F[4] + pr * u
            if nf == 6:
                C.append(r * ei)
                F.append(r * ei * u)
            return torch.stack(C), torch.stack(F), u + cs, u - cs
        (CL, FL, lpl, lml), (CR, FR, lpr, lmr) = side(L), side(R)
        ap = torch.maximum(lpl, lpr).clamp_min(0)
        am = torch.maximum(-lml, -lmr).clamp_min(0)
        F = (ap * FL + am * FR - ap * am * (CR - CL)) / (ap + am)
        faces.append(F)
        dU.narrow(t, ng, na).sub_((F.narrow(t, 1, na) - F.narrow(t, 0, na)) * dtdx)
    return faces, dU


def _ref_fill(U, ng):
    U = U.clone()
    for t in (1, 2, 3):
        n = U.shape[t]
        U.narrow(t, 0, ng).copy_(U.narrow(t, n - 2 * ng, ng).clone())
        U.narrow(t, n - ng, ng).copy_(U.narrow(t, ng, ng).clone())
    return U


def _ref_muscl(c, U):
    dt, ng = _muscl_dt(c), c["ng"]
    rec = None
    for _ in range(c["steps"]):
        F1, d1 = _ref_muscl_fluxes(_ref_fill(U, ng) if c["bc"] else U, c, dt)
        U1 = U + d1
        if c["bc"]:
            U1 = _ref_fill(U1, ng)
        F2, d2 = _ref_muscl_fluxes(U1, c, dt)
        U = 0.5 * (U + U1 + d2)
        if c["dual"]:
            v = U[1:4] / U[0]
            v2 = (v * v).sum(0)
            e, dual = U[4] / U[0] - 0.5 * v2, U[5] / U[0]
            cs2 = torch.where(e > 0, 1.4 * 0.4 * e, torch.zeros_like(e))
            e = torch.where((cs2 > 1e-3 * v2) & (e > 0.5 * dual), e, dual).clamp_min(1e-10)
            U = torch.cat([U[:4], (U[0] * (e + 0.5 * v2))[None], (U[0] * e)[None]])
        rec = [0.5 * (a + b) for a, b in zip(F1, F2)]
    if not c["record"]:
        return U
    sc = dt * (1.0 / max(c["nx"], c["ny"], c["nz"])) ** 2
    out = []
    for d in range(3):
        F = sc * rec[d][:5]
        t = 3 - d
        for o in (1, 2, 3):
            if o != t:
                F = F.narrow(o, ng, F.shape[o] - 2 * ng)
        na = F.shape[t] - 1
        planes = torch.stack([F.select(t, 0), F.select(t, na)])
        out.append([planes, F.narrow(t, 1, na - 1).movedim(t, 3).contiguous()])
    return {"state": U, "fluxes": out}


def _rounded(U, c):
    return U.float().double() if c.get("f32") else U


def exact(c, seed):
    kind = c["kind"]
    if kind in ("blocks", "amr"):
        return None   # the composite meshes' face walk has no short plain form
    with torch.no_grad():
        if kind == "grid":
            U = _rounded(_grid_state(c, seed), c)
            bcs, w = _codes(c), [1.0 / n for n in (c["nx"], c["ny"], c["nz"])[:c["rank"]]]
            for _ in range(c["steps"]):
                U = _ref_step(U, _ref_dt(U, GAMMA, w, 0.3), GAMMA, bcs, w)
            return U
        if kind == "tube":
            U = _rounded(torch.from_numpy(_tube_state(c, seed)), c)
            torch.set_num_threads(1)
            t, bcs, w = 0.0, [(c["bc"], c["bc"])], [1.0 / c["nx"]]
            while t < 0.2 * (1 - 1e-12):
                dt = min(_ref_dt(U, GAMMA, w, 0.4), 0.2 - t)
                U = _ref_step(U, dt, GAMMA, bcs, w)
                t += dt
            return U
        if kind == "gravity":
            U = _rounded(_gravity_state(c, seed), c)
            bcs, w, per = _codes(c), [1.0 / c["nx"], 1.0 / c["ny"], 1.0 / c["nz"]], c["bc"] == "periodic"
            for _ in range(c["steps"]):
                phi = _poisson(U[0], w, per)
                dt = _ref_dt(U, GAMMA, w, 0.3, 4 * math.pi)
                src = _gravity_source(phi, w, per)
                U = _ref_step(U, dt, GAMMA, bcs, w, src)
            return {"state": U, "phi": phi}
        if kind == "muscl":
            return _ref_muscl(c, _rounded(_muscl_state(c, seed), c))
        if kind == "faces":
            WL, WR, axis = [torch.from_numpy(a).cuda() for a in _face_states(c, seed)]
            F = torch.empty(WL.shape, dtype=torch.float64, device="cuda")
            for d in range(3):
                on = axis == d + 1
                F[on] = _hllc(WL[on].double().T, WR[on].double().T, GAMMA, d).T
            return F
        if kind == "rollout":
            U = _grid_state(dict(c, rank=2, nz=1), seed)
            w = torch.randn(U.shape, dtype=torch.float64, device="cuda", generator=_gen(seed))
            bcs, h, cfl = [("periodic", "periodic")] * 2, [1.0 / c["nx"], 1.0 / c["ny"]], 0.4
            states, dts = [], []
            for _ in range(c["steps"]):
                dts.append(_ref_dt(U, GAMMA, h, cfl))
                states.append(U)
                U = _ref_step(U, dts[-1], GAMMA, bcs, h)
        else:
            U = _grid_state(c, seed)
            w = torch.randn(U.shape, dtype=torch.float64, device="cuda", generator=_gen(seed))
            n = (c["nx"], c["ny"], c["nz"])[:c["rank"]]
            bcs, h, states, dts = _codes(c), [1.0 / k for k in n], [U], [0.1 / max(n)]
    for X, dt in zip(reversed(states), reversed(dts)):
        X = X.detach().requires_grad_(True)
        w, = torch.autograd.grad(_ref_step(X, dt, GAMMA, bcs, h), X, w)
    return {"final": U, "gradient": w} if kind == "rollout" else w
