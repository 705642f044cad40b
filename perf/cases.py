"""What a program built on fopis_amd spends its time on, as timed cases.

Every case goes through the package's public entry points (Host, Context,
Guess, conv3d) the way a simulation, a training script or a resume does:

  run      a simulation through the host facade: a few RootGrid::mainLoopES
           steps with boundary injection on all six faces, then the fields a
           program writes out
  stages   the same step method by method through the C ABI, with one
           injection call, for programs that keep the reference's structure
  solve    a charge density from the host to a potential and its field
  data     particles from host arrays, sorted by cell, read back with the
           diagnostics: what a resume and a dump do
  cmatrix  the capacitance matrix of a new spacecraft
  guess    the learned guess for a charge density already on the device
  grad     loss and parameter gradient of one training pair
  conv     one network layer on host buffers, forward and backward

Grid axes have m * 2^k + 1 nodes, which the multigrid coarsens; sizes, species
and options are those of fopis_amd/configs, the tests and bench.py.
"""
from __future__ import annotations

import json
import math
import os
import tempfile

import numpy as np

from fopis_amd import guess as G
from fopis_amd import lib as F
from fopis_amd import voxel_obj
from fopis_amd.host import Host

CONFIGS = os.path.join(os.path.dirname(os.path.abspath(F.__file__)), "configs")
PREC = {"fp64": F.FP64, "fp32": F.FP32}


def listed():
    return [
        # c1.json as it stands: the smallest simulation, every launch counts
        {"name": "run_33_fp64", "kind": "run", "config": "c1", "nx": 33, "ny": 33, "nz": 33, "ppc": 20,
         "box": 0, "steps": 10},
        # c2.json: the ordinary one, FP64 particles around a floating 16^3 cube
        {"name": "run_129_fp64", "kind": "run", "config": "c2", "nx": 129, "ny": 129, "nz": 129, "ppc": 64,
         "box": 16, "steps": 5},
        # c3.json at the particle count of c1.json: the largest grid, FP32, magnetised, 32^3 cube (6146 surface nodes)
        {"name": "run_257_fp32", "kind": "run", "config": "c3", "nx": 257, "ny": 257, "nz": 257, "ppc": 20,
         "box": 32, "steps": 10},
        # c5.json on an uneven grid: a photoemitting spacecraft, three species
        {"name": "run_97x81x113_photo", "kind": "run", "config": "c5", "nx": 97, "ny": 81, "nz": 113, "ppc": 16,
         "box": 8, "steps": 8},
        # the step method by method, FP64, no conductor
        {"name": "stages_65_fp64", "kind": "stages", "nx": 65, "ny": 65, "nz": 65, "ppc": 16, "precision": "fp64"},
        # a potential for a given charge: the smallest grid of the tests, FP64 multigrid
        {"name": "solve_17_fp64", "kind": "solve", "nx": 17, "ny": 17, "nz": 17, "precision": "fp64"},
        # and an uneven one with FP32 V-cycles
        {"name": "solve_129x97x161", "kind": "solve", "nx": 129, "ny": 97, "nz": 161, "precision": "fp32"},
        # a resume's particles in, sorted by cell, and out
        {"name": "data_49_fp64", "kind": "data", "nx": 49, "ny": 41, "nz": 57, "n": 1_000_003, "precision": "fp64"},
        # the capacitance matrix of c2.json's cube (1538 surface nodes)
        {"name": "cmatrix_129_cube16", "kind": "cmatrix", "nx": 129, "ny": 129, "nz": 129, "b0": 16, "b1": 16,
         "b2": 16},
        # the learned guess at the size it is trained for
        {"name": "guess_129", "kind": "guess", "nx": 129, "ny": 129, "nz": 129},
        # a training pair at the size of the quick recipes
        {"name": "grad_65", "kind": "grad", "nx": 65, "ny": 65, "nz": 65, "loss": 0},
        # a decoder layer alone: 48 -> 32 channels on an upsampled 32^3 input
        {"name": "conv_64_up_48_32", "kind": "conv", "n0": 64, "n1": 64, "n2": 64, "cin": 48, "cout": 32, "up": 1},
    ]


def _axis(rng, lo, hi):
    """A node count m * 2^k + 1 in [lo, hi], spread over the logarithm."""
    want = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    k = rng.choice([2, 3, 4])
    return max(lo, min(hi, int(max(1, round((want - 1) / 2 ** k))) * 2 ** k + 1))


def draw(rng):
    kind = rng.choice(["run", "run", "run", "stages", "solve", "data", "cmatrix", "guess", "grad", "conv"])
    if kind == "run":
        config = rng.choice(["c1", "c2", "c3", "c5"])
        nx, ny, nz = (_axis(rng, 33, 161) for _ in range(3))
        most = 64 * 128 ** 3 // (nx * ny * nz)
        return {"kind": "run", "config": config, "nx": nx, "ny": ny, "nz": nz,
                "ppc": max(4, min(most, int(math.exp(rng.uniform(math.log(8), math.log(65)))))),
                "box": 0 if config == "c1" else rng.choice([4, 6, 9, 12]), "steps": rng.randint(4, 10)}
    if kind == "stages":
        return {"kind": "stages", "nx": _axis(rng, 17, 97), "ny": _axis(rng, 17, 97), "nz": _axis(rng, 17, 97),
                "ppc": rng.randint(4, 32), "precision": rng.choice(["fp64", "fp32"])}
    if kind == "solve":
        return {"kind": "solve", "nx": _axis(rng, 17, 161), "ny": _axis(rng, 17, 161), "nz": _axis(rng, 17, 161),
                "precision": rng.choice(["fp64", "fp32"])}
    if kind == "data":
        return {"kind": "data", "nx": _axis(rng, 17, 97), "ny": _axis(rng, 17, 97), "nz": _axis(rng, 17, 97),
                "n": int(math.exp(rng.uniform(math.log(3e3), math.log(2e6)))),
                "precision": rng.choice(["fp64", "fp32"])}
    if kind == "cmatrix":
        return {"kind": "cmatrix", "nx": _axis(rng, 41, 129), "ny": _axis(rng, 41, 129), "nz": _axis(rng, 41, 129),
                "b0": rng.randint(2, 17), "b1": rng.randint(2, 17), "b2": rng.randint(2, 17)}
    if kind == "guess":
        return {"kind": "guess", "nx": _axis(rng, 17, 129), "ny": _axis(rng, 17, 129), "nz": _axis(rng, 17, 129)}
    if kind == "grad":
        return {"kind": "grad", "nx": _axis(rng, 17, 97), "ny": _axis(rng, 17, 97), "nz": _axis(rng, 17, 97),
                "loss": rng.choice([0, 1])}
    up = rng.choice([0, 1])
    n = [2 * rng.randint(5, 40) if up else rng.randint(9, 81) for _ in range(3)]
    return {"kind": "conv", "n0": n[0], "n1": n[1], "n2": n[2], "cin": rng.choice([16, 32, 48, 64]),
            "cout": rng.choice([16, 32, 48, 64]), "up": up}


# ------------------------------------------------------------------ inputs

_cache_dir = None


def _cmatrix_dir():
    """A directory for the facade's capacitance-matrix files (one per spacecraft and grid), kept by a program between
    its simulations."""
    global _cache_dir
    if _cache_dir is None:
        _cache_dir = tempfile.mkdtemp(prefix="cmatrix_")
    return _cache_dir


def _plasma(case):
    """The repository's configuration with the case's grid, particles per cell and cube, and every face injecting."""
    with open(os.path.join(CONFIGS, case["config"] + ".json")) as f:
        cfg = json.load(f)
    env = cfg["Environment"]
    env["nx"], env["ny"], env["nz"] = case["nx"], case["ny"], case["nz"]
    for sp in cfg["Plasma"].values():
        sp["particle_per_cell"] = case["ppc"]
        if sp["type"] == "ambient":
            sp["injection_axis"] = [True] * 6
    return cfg


def _box_cells(b):
    """Cells [-b/2, b - b/2) around the grid's centre."""
    return [-(x // 2) for x in b], [x - x // 2 for x in b]


def _run_state(case, seed):
    cfg = _plasma(case)
    with tempfile.TemporaryDirectory() as d:
        if case["box"]:
            lo, hi = _box_cells([case["box"]] * 3)
            obj = os.path.join(d, "box.obj")
            voxel_obj.write_boxes(obj, [(tuple(lo), tuple(hi))])
            cfg["Object"]["Spacecraft"]["file_name"] = obj
        else:
            cfg["Object"] = {}
        path = os.path.join(d, "input.json")
        with open(path, "w") as f:
            json.dump(cfg, f)
        h = Host(path, device_loader=True, device_seed=1000 + seed, device_injection=True,
                 cmatrix_cache=_cmatrix_dir() if case["box"] else "")
    return {"host": h, "steps": case["steps"], "object": bool(case["box"])}


def _run(state):
    h, ctx = state["host"], state["host"].ctx
    for _ in range(state["steps"]):
        h.main_loop_es()
    out = {"phi": ctx.get_field(F.PHI), "rho": ctx.get_field(F.RHO, 0),
           "density": [ctx.get_field(F.DENSITY, s) for s in range(2)], "energy": list(ctx.energy()),
           "particles": [ctx.num_particles(s) for s in range(ctx.S)]}
    if state["object"]:
        st = ctx.object_state(0)
        out["potential"], out["current"], out["surface"] = st["potential"], st["current"], st["charge_map"]
    return out


_SPECIES = [(-1.0, 1.0, 4.0), (1.0, 100.0, 4.0)]  # charge, mass, particles per superparticle
_SIGMA = (0.1, 0.01)  # thermal speeds in cells per step
_EPS0 = 6400.0


def _stages_state(case, seed):
    n = (case["nx"], case["ny"], case["nz"])
    ctx = F.Context(F.make_desc(*n, _SPECIES, _EPS0, static_b=(0.0, 0.0, 0.2), precision=PREC[case["precision"]],
                                mg_precision=F.FP32))
    hi = [v - 1.0 for v in n]
    counts = []
    for s in range(2):
        ctx.load_maxwellian(s, case["ppc"] * math.prod(v - 1 for v in n), 100 * seed + s, [0.0] * 3, hi, [0.0] * 3,
                            _SIGMA[s])
        # the one-way flux of a Maxwellian through each face
        flux = case["ppc"] * _SIGMA[s] / math.sqrt(2 * math.pi)
        counts.append([int(flux * hi[(a + 1) % 3] * hi[(a + 2) % 3]) for a in (0, 0, 1, 1, 2, 2)])
    ctx.initialize()
    return {"ctx": ctx, "counts": counts, "seed": 7919 * seed, "step": 0}


def _stages(state):
    ctx = state["ctx"]
    state["step"] += 1
    ctx.update_particle_velocity_es()
    ctx.update_particle_position_es()
    for s in range(2):
        ctx.inject_maxwellian(s, state["counts"][s], state["seed"] + 2 * state["step"] + s, [0.0] * 3, _SIGMA[s],
                              _SIGMA[s])
    ctx.update_density()
    ctx.update_rho()
    ctx.solve_poisson()
    ctx.update_efield()
    return {"phi": ctx.get_field(F.PHI), "rho": ctx.get_field(F.RHO, 0), "density": ctx.get_field(F.DENSITY, 0),
            "ex": ctx.get_field(F.EXREF), "energy": list(ctx.energy())}


def _charge(shape, seed, nodes):
    """A node charge density in the glue layout: a smooth structure of random blobs plus particle noise, at the
    interior nodes."""
    rng = np.random.default_rng(seed)
    rho = np.zeros(shape)
    x = [np.linspace(0.0, 1.0, n) for n in nodes]
    r = 0.5 * rng.standard_normal([n - 2 for n in nodes])
    for _ in range(4):
        c, w = rng.uniform(0.2, 0.8, 3), rng.uniform(0.05, 0.2)
        g = [np.exp(-((x[a][1:-1] - c[a]) / w) ** 2) for a in range(3)]
        r += 3.0 * rng.standard_normal() * g[0][:, None, None] * g[1][None, :, None] * g[2][None, None, :]
    rho[2:-2, 2:-2, 2:-2] = r
    return rho


def _solve_inputs(case, seed):
    n = (case["nx"], case["ny"], case["nz"])
    return n, _charge(tuple(v + 2 for v in n), seed, n)


def _solve_state(case, seed):
    n, rho = _solve_inputs(case, seed)
    ctx = F.Context(F.make_desc(*n, _SPECIES[:1], 1.0, precision=PREC[case["precision"]]))
    return {"ctx": ctx, "rho": rho, "zero": np.zeros_like(rho)}


def _solve(state):
    ctx = state["ctx"]
    ctx.set_field(F.RHO, state["rho"])
    ctx.set_field(F.PHI, state["zero"])
    ctx.solve_poisson()
    ctx.update_efield()
    return {"phi": ctx.get_field(F.PHI), "e": [ctx.get_field(w) for w in (F.EXREF, F.EYREF, F.EZREF)]}


def _dst_solve(n, rho):
    from scipy.fft import dstn, idstn

    lam = [2.0 - 2.0 * np.cos(np.pi * np.arange(1, v - 1) / (v - 1)) for v in n]
    lam = lam[0][:, None, None] + lam[1][None, :, None] + lam[2][None, None, :]
    phi = np.zeros_like(rho)
    phi[2:-2, 2:-2, 2:-2] = idstn(dstn(rho[2:-2, 2:-2, 2:-2], type=1) / lam, type=1)
    return phi


def _solve_exact(case, seed):
    n, rho = _solve_inputs(case, seed)
    phi = _dst_solve(n, rho)
    e = []
    for a in range(3):
        # nodal field inside the domain: central differences, one-sided of second order at the faces
        p = np.moveaxis(phi[1:-1, 1:-1, 1:-1], a, 0)
        q = np.empty_like(p)
        q[1:-1] = 0.5 * (p[:-2] - p[2:])
        q[0] = 0.5 * (p[2] - 4.0 * p[1] + 3.0 * p[0])
        q[-1] = 0.5 * (-p[-3] + 4.0 * p[-2] - 3.0 * p[-1])
        f = np.zeros_like(phi)
        f[1:-1, 1:-1, 1:-1] = np.moveaxis(q, 0, a)
        e.append(f)
    return {"phi": phi, "e": e}


def _data_inputs(case, seed):
    rng = np.random.default_rng(seed)
    hi = [case["nx"] - 1.0, case["ny"] - 1.0, case["nz"] - 1.0]
    sets = []
    for s in range(2):
        d = {k: rng.uniform(0.0, hi[a], case["n"]) for a, k in enumerate("xyz")}
        d.update({k: rng.normal(0.0, _SIGMA[s], case["n"]) for k in ("vx", "vy", "vz")})
        sets.append(d)
    return sets


def _data_state(case, seed):
    n = (case["nx"], case["ny"], case["nz"])
    ctx = F.Context(F.make_desc(*n, _SPECIES, _EPS0, precision=PREC[case["precision"]]))
    return {"ctx": ctx, "sets": _data_inputs(case, seed)}


def _data(state):
    ctx = state["ctx"]
    for s, d in enumerate(state["sets"]):
        ctx.set_particles(s, d)
    ctx.sort_by_cell()
    out = []
    for s in range(2):
        m = ctx.moments(s)
        out.append({"particles": ctx.get_particles(s), "mean_x": m["mean_x"], "mean_v": m["mean_v"],
                    "var_v": m["var_v"]})
    return {"species": out, "kinetic": ctx.energy()[0]}


def _data_exact(case, seed):
    t = [-(-(case[k] - 1) // 8) for k in ("nx", "ny", "nz")]
    out, kinetic = [], 0.0
    for s, d in enumerate(_data_inputs(case, seed)):
        if case["precision"] == "fp32":  # the cells of the rounded positions order the particles
            d = {k: v.astype(np.float32).astype(np.float64) for k, v in d.items()}
        c = [np.minimum(np.floor(d[k]).astype(np.int64), case["n" + k] - 2) for k in "xyz"]
        key = ((c[0] // 8 * t[1] + c[1] // 8) * t[2] + c[2] // 8) * 512 + ((c[0] % 8) * 8 + c[1] % 8) * 8 + c[2] % 8
        order = np.argsort(key, kind="stable")
        d = {k: v[order] for k, v in d.items()}
        v = np.stack([d[k] for k in ("vx", "vy", "vz")])
        kinetic += 0.5 * _SPECIES[s][1] * _SPECIES[s][2] * (v * v).sum()
        out.append({"particles": d, "mean_x": np.array([d[k].mean() for k in "xyz"]), "mean_v": v.mean(1),
                    "var_v": v.var(1)})
    return {"species": out, "kinetic": float(kinetic)}


def _box_nodes(case, seed):
    """A box conductor near the grid's centre: its cell map and surface nodes in the glue layout."""
    rng = np.random.default_rng(seed)
    n = [case["nx"], case["ny"], case["nz"]]
    b = [case["b0"], case["b1"], case["b2"]]
    lo = [v // 2 - w // 2 + int(rng.integers(-3, 4)) for v, w in zip(n, b)]
    mask = np.zeros([v + 1 for v in n], np.uint8)
    mask[tuple(slice(p, p + w) for p, w in zip(lo, b))] = 1
    ax = [np.arange(p, p + w + 1) for p, w in zip(lo, b)]
    i, j, k = (v.ravel() for v in np.meshgrid(*ax, indexing="ij"))
    on = np.zeros(i.shape, bool)
    for v, p, w in zip((i, j, k), lo, b):
        on |= (v == p) | (v == p + w)
    return mask, np.stack([i, j, k], 1)[on].astype(np.int32)


def _cmatrix_state(case, seed):
    ctx = F.Context(F.make_desc(case["nx"], case["ny"], case["nz"], _SPECIES, 1.0, mg_precision=F.FP32))
    mask, nodes = _box_nodes(case, seed)
    return {"ctx": ctx, "mask": mask, "nodes": nodes}


def _cmatrix(state):
    ctx = state["ctx"]
    ctx.set_object(0, state["mask"], state["nodes"])
    ctx.build_cmatrix(0)
    return ctx.get_cmatrix(0)


def _cmatrix_exact(case, seed):
    """The inverse of the discrete Green's function between the surface nodes, by sine transforms."""
    import torch

    _, nodes = _box_nodes(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    S, L = [], []
    for a, v in enumerate((case["nx"], case["ny"], case["nz"])):
        m, u = v - 2, nodes[:, a] - 1
        k = np.arange(1, m + 1)
        S.append(torch.from_numpy(np.sqrt(2.0 / (m + 1)) * np.sin(np.pi * np.outer(u, k) / (m + 1))).to(dev))
        L.append(torch.from_numpy(4.0 * np.sin(np.pi * k / (2.0 * (m + 1))) ** 2).to(dev))
    B = torch.zeros((len(nodes), len(nodes)), dtype=torch.float64, device=dev)
    for k in range(len(L[0])):
        # the two remaining axes at once: sum over (l, m) of products of node pairs
        inv = 1.0 / (L[0][k] + L[1][:, None] + L[2][None, :])
        w = (S[1][:, :, None] * S[2][:, None, :]).reshape(len(nodes), -1) * S[0][:, k][:, None]
        B += (w * inv.reshape(1, -1)) @ w.t()
    return torch.linalg.inv(B).cpu().numpy()


def _params(seed):
    """Network parameters of the layers' shapes: He-normal kernels, small biases."""
    rng = np.random.default_rng(seed)
    slices, total = G.param_slices()
    p = np.zeros(total, np.float32)
    for name, ws, shape, bs in slices:
        w = rng.standard_normal(shape) * math.sqrt(2.0 / (27 * (2 if name == "e0a" else shape[1])))
        p[ws] = w.astype(np.float32).ravel()
        p[bs] = (0.05 * rng.standard_normal(shape[2])).astype(np.float32)
    return p


def _guess_state(case, seed):
    n = (case["nx"], case["ny"], case["nz"])
    ctx = F.Context(F.make_desc(*n, _SPECIES[:1], 1.0, mg_precision=F.FP32))
    g = G.Guess(ctx)
    g.set_params(_params(seed), 2.0)
    ctx.set_field(F.RHO, _charge(ctx.field_shape(F.RHO), seed, n))
    return {"ctx": ctx, "guess": g}


def _guess(state):
    # the guess twice, as for the two solves of a step, then the potential
    state["guess"].apply()
    state["guess"].apply()
    return state["ctx"].get_field(F.PHI)


def _bf16(t):
    import torch

    return t.to(torch.float32).to(torch.bfloat16).to(t.dtype)


def _net(x, params, dev):
    """The network on [n0, n1, n2, 8] in 64 bits, weights rounded to BF16 as the device holds them."""
    import torch

    slices, _ = G.param_slices()
    layer = {}
    for (name, ws, shape, bs), (_, _, _, up, relu) in zip(slices, G.LAYERS):
        layer[name] = (_bf16(params[ws].reshape(shape)), params[bs], up, relu)

    def conv(name, x, skip=None):
        w, b, up, relu = layer[name]
        if up:
            for a in range(3):
                x = x.repeat_interleave(2, dim=a)
        n = x.shape[:3]
        xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
        y = b.expand(n + (w.shape[2],))
        for t in range(27):
            i, j, k = t // 9, t // 3 % 3, t % 3
            y = y + xp[i:i + n[0], j:j + n[1], k:k + n[2]].reshape(-1, x.shape[3]).matmul(w[t]).reshape(y.shape)
        if skip is not None:
            y = y + skip
        return torch.relu(y) if relu else y

    def pool(x):
        a, b, c, q = x.shape
        return x.reshape(a // 2, 2, b // 2, 2, c // 2, 2, q).mean((1, 3, 5))

    s0 = conv("e0b", conv("e0a", x))
    s1 = conv("e1b", conv("e1a", pool(s0)))
    s2 = conv("e2b", conv("e2a", pool(s1)))
    b3 = conv("e3b", conv("e3a", pool(s2)))
    e2 = conv("d2b", conv("d2a", b3, s2))
    e1 = conv("d1b", conv("d1a", e2, s1))
    return conv("out", conv("d0b", conv("d0a", e1, s0)))[..., 0]


def _features(rho_hat, mask=None):
    import torch

    x = torch.zeros(tuple(rho_hat.shape) + (8,), dtype=torch.float64, device=rho_hat.device)
    x[..., 0] = rho_hat
    if mask is not None:
        x[..., 1] = mask
    return x


def _guess_exact(case, seed):
    import torch

    dev = "cuda" if torch.cuda.is_available() else "cpu"
    n = (case["nx"], case["ny"], case["nz"])
    rho = _charge(tuple(v + 2 for v in n), seed, n)
    inner = rho[2:-2, 2:-2, 2:-2]
    sigma = math.sqrt((inner * inner).mean())
    r = torch.zeros(G.net_grid(*n), dtype=torch.float64, device=dev)
    r[:n[0] - 2, :n[1] - 2, :n[2] - 2] = torch.from_numpy(inner / sigma).to(dev)
    with torch.no_grad():
        out = _net(_features(_bf16(r)), torch.from_numpy(_params(seed)).to(dev, torch.float64), dev)
    phi = np.zeros_like(rho)
    phi[2:-2, 2:-2, 2:-2] = out[:n[0] - 2, :n[1] - 2, :n[2] - 2].cpu().numpy() * 2.0 * sigma
    return phi


def _grad_inputs(case, seed):
    n = (case["nx"], case["ny"], case["nz"])
    grid = G.net_grid(*n)
    rho = _charge(tuple(v + 2 for v in n), seed, n)
    phi = _dst_solve(n, rho)[2:-2, 2:-2, 2:-2]
    rho = rho[2:-2, 2:-2, 2:-2]
    sigma = math.sqrt((rho * rho).mean())
    r, p = np.zeros(grid, np.float32), np.zeros(grid, np.float32)
    inside = tuple(slice(0, v - 2) for v in n)
    r[inside], p[inside] = rho / sigma, phi / sigma
    mask = np.zeros(grid, np.uint8)
    c = [v // 2 for v in n]
    mask[c[0] - 3:c[0] + 3, c[1] - 3:c[1] + 3, c[2] - 3:c[2] + 3] = 1
    return G.to_bf16(r), mask, G.to_bf16(p), inside


def _grad_state(case, seed):
    n = (case["nx"], case["ny"], case["nz"])
    ctx = F.Context(F.make_desc(*n, _SPECIES[:1], 1.0, mg_precision=F.FP32))
    g = G.Guess(ctx)
    r, mask, p, _ = _grad_inputs(case, seed)
    g.set_params(_params(seed), float(np.sqrt(np.mean(G.from_bf16(p) ** 2))))
    g.set_loss(case["loss"])
    g.dataset_alloc(1)
    g.dataset_set(0, r, mask, p)
    return {"ctx": ctx, "guess": g}


def _grad(state):
    loss, grad = state["guess"].grad(0)
    return {"loss": loss, "grad": grad}


def _grad_exact(case, seed):
    import torch

    if math.prod(case[k] for k in ("nx", "ny", "nz")) > 70 ** 3:
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    r, mask, p, inside = _grad_inputs(case, seed)
    scale = float(np.sqrt(np.mean(G.from_bf16(p) ** 2)))
    params = torch.from_numpy(_params(seed)).to(dev, torch.float64).requires_grad_(True)
    r, p = (torch.from_numpy(G.from_bf16(v).astype(np.float64)).to(dev) for v in (r, p))
    out = _net(_features(r, torch.from_numpy(mask.astype(np.float64)).to(dev)), params, dev)[inside]
    if case["loss"]:
        u = torch.nn.functional.pad(out, (1, 1, 1, 1, 1, 1))
        au = 6.0 * out - (u[:-2, 1:-1, 1:-1] + u[2:, 1:-1, 1:-1] + u[1:-1, :-2, 1:-1] + u[1:-1, 2:, 1:-1] +
                          u[1:-1, 1:-1, :-2] + u[1:-1, 1:-1, 2:])
        d = scale * au - r[inside]
    else:
        d = out - p[inside] / scale
    loss = 0.5 * (d * d).mean()
    loss.backward()
    return {"loss": float(loss.detach()), "grad": params.grad.cpu().numpy()}


def _conv_state(case, seed):
    rng = np.random.default_rng(seed)
    n = (case["n0"], case["n1"], case["n2"])
    xs = tuple(v // 2 for v in n) if case["up"] else n
    return {"x": G.to_bf16(np.maximum(rng.standard_normal(xs + (case["cin"],), np.float32), 0.0)),
            "w": (rng.standard_normal((27, case["cin"], case["cout"]), np.float32) * 0.05),
            "b": rng.standard_normal(case["cout"]).astype(np.float32),
            "add": G.to_bf16(rng.standard_normal(n + (case["cout"],), np.float32)),
            "g": G.to_bf16(rng.standard_normal(n + (case["cout"],), np.float32)), "up": bool(case["up"])}


def _conv(state):
    y = G.conv3d(state["x"], state["w"], state["b"], up=state["up"], relu=True, add_bf16=state["add"])
    dw, db, dx = G.conv3d_backward(state["x"], state["w"], state["g"], up=state["up"])
    return {"y": y, "dw": dw, "db": db, "dx": dx}


def _conv_exact(case, seed):
    import torch

    dev = "cuda" if torch.cuda.is_available() else "cpu"
    s = _conv_state(case, seed)
    x, g = (torch.from_numpy(G.from_bf16(s[k]).astype(np.float64)).to(dev) for k in ("x", "g"))
    if s["up"]:
        for a in range(3):
            x = x.repeat_interleave(2, dim=a)
    n = x.shape[:3]
    xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
    g = g.reshape(-1, case["cout"])
    dw = [xp[t // 9:t // 9 + n[0], t // 3 % 3:t // 3 % 3 + n[1], t % 3:t % 3 + n[2]].reshape(-1, case["cin"]).t() @ g
          for t in range(27)]
    return {"y": None, "dw": torch.stack(dw).cpu().numpy(), "db": g.sum(0).cpu().numpy(), "dx": None}


# ------------------------------------------------------------------ the interface

_PREPARE = {"run": _run_state, "stages": _stages_state, "solve": _solve_state, "data": _data_state,
            "cmatrix": _cmatrix_state, "guess": _guess_state, "grad": _grad_state, "conv": _conv_state}
_RUN = {"run": _run, "stages": _stages, "solve": _solve, "data": _data, "cmatrix": _cmatrix, "guess": _guess,
        "grad": _grad, "conv": _conv}
_EXACT = {"solve": _solve_exact, "data": _data_exact, "cmatrix": _cmatrix_exact, "guess": _guess_exact,
          "grad": _grad_exact, "conv": _conv_exact}


def prepare(case, seed):
    return dict(_PREPARE[case["kind"]](case, seed), kind=case["kind"])


def run(state):
    return _RUN[state["kind"]](state)


def exact(case, seed):
    f = _EXACT.get(case["kind"])  # a simulation drawn on the device has no such value
    return f(case, seed) if f else None


def work(case):
    kind = case["kind"]
    if kind == "conv":
        nv = case["n0"] * case["n1"] * case["n2"]
        nin = nv // 8 if case["up"] else nv
        ci, co = case["cin"], case["cout"]
        # forward, weight gradient and data gradient are one product each; x, the addend and the gradient in, y and dx out
        return {"bytes": 2.0 * (2 * nin * ci + nv * (3 * co + ci)) + 8.0 * 27 * ci * co,
                "flops": 3 * 2.0 * 27 * ci * co * nv}
    n = case["nx"] * case["ny"] * case["nz"]
    if kind in ("run", "stages"):
        pb = 48 if case.get("precision") == "fp32" or case.get("config") in ("c3", "c5") else 96
        steps, ppc = case.get("steps", 1), case["ppc"]
        # every particle's six components in and out, and the fields: rho of each species, phi in and out, E
        return {"bytes": steps * n * (2.0 * ppc * pb + 8 * 8) + 4 * 8.0 * n,
                "flops": steps * n * (2.0 * ppc * 250 + 200)}
    if kind == "solve":
        return {"bytes": 6 * 8.0 * n, "flops": 300.0 * n}
    if kind == "data":
        return {"bytes": 2 * 2 * 48.0 * case["n"], "flops": 2 * 30.0 * case["n"]}
    if kind == "cmatrix":
        b = [case["b0"] + 1, case["b1"] + 1, case["b2"] + 1]
        m = math.prod(b) - math.prod(v - 2 for v in b)
        return {"bytes": 2 * 8.0 * m * m, "flops": 2.0 * m ** 3}
    grid = [v for v in G.net_grid(case["nx"], case["ny"], case["nz"])]
    nv = math.prod(grid)
    flops = sum(2.0 * 27 * ci * co * nv / 8 ** lvl for ci, co, lvl, _, _ in G.LAYERS)
    act = sum(2.0 * (ci / (8 if up else 1) + co) * nv / 8 ** lvl for ci, co, lvl, up, _ in G.LAYERS)
    if kind == "guess":
        return {"bytes": 2 * (act + 16.0 * n) + 8.0 * n, "flops": 2 * flops}
    return {"bytes": 3 * act + 5.0 * nv, "flops": 3 * flops}
