"""Timed cases: what a program that uses this framework has it do, through its public entry points.

A simulation asks for one Newton linear solve after another (``scene.minimizeEnergy``: the
energies' gradients and projected Hessians, assembly, PCG) on meshes from a thousand to a
million and a half tets, with block-Jacobi or MAS, in FP64 or with FP32 values and FP64
refinement; with contact its pair sets change on every step. Around the solve it evaluates
energies alone, multiplies with the assembled Hessian, bounds its steps by continuous
collision detection, differentiates an equilibrium with respect to its material, or serves
the solves of many clients in batches. Sizes are those of the configurations, tests and
benchmark of this repository, and odd ones between them.
"""
from __future__ import annotations

import dataclasses
import functools
import math
import os
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

# ------------------------------------------------------------------------------ the cases


def listed():
    return [
        # the smallest solve: the 8^3-cell cube to 1e-8, bound by latency and launches
        {"name": "newton_n8_jacobi", "kind": "newton", "n": 8, "solver": "jacobian",
         "precision": "fp64", "tol": 1e-8, "young": 1e5},
        # a client's request of the serving stream solved alone with its preconditioner, odd size
        {"name": "newton_n17_mas_mixed", "kind": "newton", "n": 17, "solver": "mas",
         "precision": "mixed", "tol": 1e-6, "young": 3e5},
        # the ordinary solve of an animation step, FP32 values and FP64 refinement
        {"name": "newton_n31_jacobi_mixed", "kind": "newton", "n": 31, "solver": "jacobian",
         "precision": "mixed", "tol": 1e-6, "young": 1e5},
        # the benchmark's solve: 663,552 tets, FP64, block-Jacobi
        {"name": "newton_n48_jacobi", "kind": "newton", "n": 48, "solver": "jacobian",
         "precision": "fp64", "tol": 1e-6, "young": 1e5},
        # the largest solve: 1,572,864 tets, an operator beyond the last-level cache
        {"name": "newton_n64_jacobi", "kind": "newton", "n": 64, "solver": "jacobian",
         "precision": "fp64", "tol": 1e-6, "young": 1e5},
        # energies alone: gradient and projected Hessian of 303,918 tets, assembled
        {"name": "assembly_n37", "kind": "assembly", "n": 37, "projection": 2, "young": 1e5},
        # cloth: StVK membrane and dihedral bending of an odd grid, assembled
        {"name": "cloth_m203", "kind": "cloth", "m": 203, "projection": 2},
        # a caller's own iteration: products with the assembled Hessian
        {"name": "spmv_n41", "kind": "spmv", "n": 41, "young": 1e5},
        # a contact step: affine and free bodies on a cloth, pairs re-indexed, 9x9 .. 3x3 blocks
        {"name": "contact_newton", "kind": "contact", "bodies_x": 3, "bodies_z": 2, "cells": 9,
         "cloth_m": 97, "pairs": 45000, "tol": 1e-4},
        # backward: the adjoint of an equilibrium with respect to per-tet stiffness
        {"name": "adjoint_n13", "kind": "adjoint", "n": 13, "tol": 1e-10},
        # the line search of a contact step: swept candidates and the step bound
        {"name": "ccd_step", "kind": "ccd", "bodies_x": 3, "bodies_z": 3, "cells": 9,
         "cloth_m": 129, "fall": 0.004},
        # continuous batching: clients' solves of mixed sizes arriving together
        {"name": "serving_burst", "kind": "serving", "count": 12, "n_min": 6, "n_max": 20},
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], even over the logarithm."""
    return max(lo, min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(["newton", "newton", "newton", "assembly", "cloth", "spmv", "contact",
                       "adjoint", "ccd", "serving"])
    young = 10.0 ** rng.uniform(4.0, 6.0)
    if kind == "newton":
        solver = rng.choice(["jacobian", "jacobian", "mas"])
        return {"kind": kind, "n": _log(rng, 6, 20 if solver == "mas" else 56), "solver": solver,
                "precision": rng.choice(["fp64", "mixed"]), "tol": rng.choice([1e-6, 1e-8]),
                "young": young}
    if kind == "assembly":
        return {"kind": kind, "n": _log(rng, 5, 48), "projection": rng.choice([0, 1, 2]),
                "young": young}
    if kind == "cloth":
        return {"kind": kind, "m": _log(rng, 17, 260), "projection": rng.choice([0, 1, 2])}
    if kind == "spmv":
        return {"kind": kind, "n": _log(rng, 5, 60), "young": young}
    if kind == "contact":
        return {"kind": kind, "bodies_x": rng.randint(1, 4), "bodies_z": rng.randint(1, 3),
                "cells": rng.randint(5, 10), "cloth_m": rng.randint(48, 128),
                "pairs": _log(rng, 5000, 60000), "tol": 1e-4}
    if kind == "adjoint":
        return {"kind": kind, "n": _log(rng, 4, 14), "tol": 1e-10}
    if kind == "ccd":
        return {"kind": kind, "bodies_x": rng.randint(1, 4), "bodies_z": rng.randint(1, 3),
                "cells": rng.randint(5, 10), "cloth_m": rng.randint(40, 160),
                "fall": rng.uniform(0.001, 0.01)}
    return {"kind": kind, "count": rng.randint(4, 14), "n_min": 6, "n_max": rng.randint(10, 22)}


# ------------------------------------------------------------------------------ inputs


@functools.lru_cache(maxsize=4)
def _cube(n):
    """Rest mesh of the n^3-cell cube (bottom fixed); positions are drawn per seed."""
    from yasps_amd.scenes import cube_scene
    return cube_scene(n, noise=0.0)


def _cube_case(case, seed):
    from yasps_amd.scenes import lame_parameters
    base = _cube(case["n"])
    rng = np.random.default_rng(seed)
    x = base.rest.copy()
    x[base.n_fixed:] += rng.normal(0.0, 0.02 / base.n, size=(base.n_moving, 3))
    mu, lam = lame_parameters(case["young"], base.poisson)
    return dataclasses.replace(base, position=x, mu=mu, lam=lam, young=case["young"])


def _cube_scene(case, seed, projection=2, solver="jacobian", **options):
    from yasps_amd.scenes import build_yasps_scene
    s0, _ = build_yasps_scene(_cube_case(case, seed), projection_method=projection,
                              solver_name=solver, **options)
    s0.minimizer.computeNumericValue()          # the static structure, built once per scene
    return s0


@functools.lru_cache(maxsize=4)
def _cloth_mesh(m):
    from yasps_amd.scenes import grid_cloth
    rest, _, tri, hinges = grid_cloth(m, 0.0, np.random.default_rng(0))
    return rest, tri, hinges


_CLOTH = {"mu": 1e3, "lam": 8e2, "thickness": 1e-3, "dt": 1e-2, "bend": 1e-4}


def _cloth_positions(m, seed):
    rest = _cloth_mesh(m)[0]
    return rest + np.random.default_rng(seed).normal(0.0, 0.05 / (m - 1), size=rest.shape)


def _cloth_scene(case, seed):
    from yasps_amd import scene, energies as en
    rest, tri, hinges = _cloth_mesh(case["m"])
    s0 = scene("cloth")
    m = s0.addMesh("sheet")
    mv = m.addPrimitive("moving_vertices", numInstances=rest.shape[0])
    mv.addAttribute("position", rows=3, cols=1).updateValue(_cloth_positions(case["m"], seed))
    mv.addConstant("rest_position", rows=3, cols=1).updateValue(rest)
    for name, conn, arity in (("triangles", tri, 3), ("hinges", hinges, 4)):
        el = m.addPrimitive(name, numInstances=conn.shape[0])
        e2v = el.addConnectivity(name + "2v", mv, conn, arity)
        pos = el.addAttribute("positions", through=e2v, source=mv["position"])
        ref = el.addAttribute("rest_positions", through=e2v, source=mv["rest_position"])
        c = _CLOTH
        energy = en.stvk_membrane(ref, pos, c["mu"], c["lam"], c["thickness"], c["dt"]) \
            if arity == 3 else en.bending(pos, ref, c["bend"])
        s0.addEnergy(el.addAttribute("energy", computed_attribute=energy),
                     projection_method=case["projection"])
    s0.addMinimizeTarget([mv["position"]])
    s0.minimizer.computeNumericValue()
    return s0


@functools.lru_cache(maxsize=4)
def _bodies(bodies_x, bodies_z, cells, cloth_m, pairs, dhat):
    from yasps_amd.scenes import contact_scene
    return contact_scene(bodies_x=bodies_x, bodies_z=bodies_z, cells=cells, cloth_m=cloth_m,
                         max_pairs=pairs, dhat=dhat)


def _contact(case, seed, pairs, dhat):
    """Bodies over a cloth and the pairs between them; the seed moves every free vertex and
    every affine body a little and gives them velocities (the pairs stay the same)."""
    base = _bodies(case["bodies_x"], case["bodies_z"], case["cells"], case["cloth_m"], pairs, dhat)
    rng = np.random.default_rng(seed)
    moving = base.n_fixed + base.n_abd
    x, v = base.position.copy(), np.zeros_like(base.velocity)
    x[moving:, [0, 2]] += rng.normal(0.0, 2e-5, size=(base.n_free, 2))
    v[base.n_fixed:] = rng.normal(0.0, 0.02, size=(v.shape[0] - base.n_fixed, 3))
    return dataclasses.replace(base, position=x, velocity=v,
                               A=base.A + 1e-3 * rng.standard_normal(base.A.shape),
                               t=base.t + 1e-6 * rng.standard_normal(base.t.shape))


def _ccd_state(case, seed):
    """Surfaces of the bodies and the cloth, every body falling (x - t d)."""
    from yasps_amd import device as dev
    from yasps_amd.ccd import CCD
    from yasps_amd.scenes import boundary_faces
    cs = _contact(case, seed, 1, 1e-5)
    x = cs.positions()
    per = cs.tets.shape[0] // (cs.n_bodies + cs.n_free_bodies)
    mesh = np.ones(x.shape[0], dtype=np.uint32)
    mesh[cs.tets.reshape(-1)] = 2 + np.repeat(np.arange(cs.tets.shape[0]) // per, 4)
    faces = np.concatenate([boundary_faces(cs.tets), cs.triangles])
    e = np.sort(np.concatenate([faces[:, [0, 1]], faces[:, [1, 2]], faces[:, [0, 2]]]), axis=1)
    edges = np.unique(e, axis=0)
    c = CCD(int(np.unique(faces).size), x.shape[0], max_cd_pairs=100_000_000,
            max_ccd_pairs=100_000_000, mesh_indices=mesh, print_timings=False)
    d = np.zeros_like(x)
    d[mesh > 1, 1] = case["fall"]
    d[mesh > 1] += np.random.default_rng(seed).normal(0.0, 0.1 * case["fall"],
                                                      size=(int((mesh > 1).sum()), 3))
    xd, dd = dev.to_device(x.reshape(-1), "float64"), dev.to_device(d.reshape(-1), "float64")
    c.init_faces(xd, faces.reshape(-1), np.unique(faces), len(faces))
    c.init_edges(xd, xd, edges.reshape(-1), len(edges))
    return {"ccd": c, "x": xd, "d": dd, "dhat": 1e-5}


def _adjoint_state(case, seed):
    """An equilibrium under gravity and the loss gradient at it."""
    from yasps_amd.adjoint import MaterialProblem
    pb = MaterialProblem(case["n"], solver="jacobian")
    rng = np.random.default_rng(seed)
    x = pb.equilibrium(math.log(1e5) + 0.3 * rng.standard_normal(pb.num_tets), tol=1e-8,
                       pcg_tol=1e-8)
    xbar = np.zeros((pb.n_free, 3))
    xbar[pb.top] = rng.normal(0.0, 1.0, size=(pb.top.size, 3))
    return {"problem": pb, "x": x, "xbar": xbar.reshape(-1)}


def _serving_state(case, seed):
    """A warm server (a slot for every request) and the clients' payloads."""
    from yasps_amd.serving import SolveServer, attach_payloads, serving_stream
    fixed = serving_stream(case["count"], case["n_min"], case["n_max"], seed=7)
    stream = serving_stream(case["count"], case["n_min"], case["n_max"], seed=seed)
    for a, b in zip(stream, fixed):
        a.n = b.n                               # the meshes a deployment serves stay the same
    server = SolveServer(max_active=case["count"], keep_solutions=True)
    sizes = [r.n for r in stream]
    for n in sorted(set(sizes)):
        server.pool[n] = [server._new_slot(n) for _ in range(sizes.count(n))]
    return {"server": server, "requests": attach_payloads(stream)}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "newton":
        options = {"threshold_mode": "relative_residual", "precision": case["precision"]}
        if case["solver"] == "mas":
            options.update(max_levels=4, coarsest_level_weight=1.0)
        s0 = _cube_scene(case, seed, solver=case["solver"], **options)
        if case["solver"] == "mas":
            h = s0.minimizer.activeHessian      # the hierarchy, built once per structure
            s0.minimizer.linearSolver.implementation._ensure(h, h.rows)
        return {"scene": s0, "tol": case["tol"]}
    if kind == "assembly":
        return {"scene": _cube_scene(case, seed, case["projection"])}
    if kind == "cloth":
        return {"scene": _cloth_scene(case, seed)}
    if kind == "spmv":
        from yasps_amd import vector
        h = _cube_scene(case, seed).minimizer.activeHessian
        return {"hessian": h, "x": vector().updateValue(_spmv_vector(h.rows, seed))}
    if kind == "contact":
        from yasps_amd.scenes import build_contact_scene
        s0, _ = build_contact_scene(_contact(case, seed, case["pairs"], 1e-3),
                                    threshold_mode="relative_residual")
        s0.minimizer.computeNumericValue()
        return {"scene": s0, "tol": case["tol"]}
    if kind == "adjoint":
        return dict(_adjoint_state(case, seed), tol=case["tol"])
    if kind == "ccd":
        return _ccd_state(case, seed)
    return _serving_state(case, seed)


def _spmv_vector(n, seed):
    return np.random.default_rng(seed + 1).standard_normal(n)


# ------------------------------------------------------------------------------ one pass


def _assembled(h):
    out = {"gradient": h.gradient.value, "hessian": h.blocks_flattened}
    if h.blocks_flattened_dynamic is not None:
        out["hessian_dynamic"] = h.blocks_flattened_dynamic
    return out


def run(state):
    if "server" in state:
        done = state["server"].serve([dataclasses.replace(r) for r in state["requests"]])
        return [r.solution for r in sorted(done, key=lambda r: r.id)]
    if "ccd" in state:
        c = state["ccd"]
        found = c.ccd(state["x"], state["dhat"], state["d"], 1.0)
        step = c.compute_largest_step_size(0.8, state["x"], state["d"])
        return {"candidates": int(found), "step": float(step)}
    if "problem" in state:
        return {"theta_gradient": state["problem"].vjp(state["x"], state["xbar"],
                                                       pcg_tol=state["tol"])}
    if "hessian" in state:
        return {"y": state["hessian"].spmv(state["x"]).value}
    if "tol" in state:
        step = state["scene"].minimizeEnergy(tolerance=state["tol"])
        return dict(_assembled(state["scene"].minimizer.activeHessian), step=list(step))
    return _assembled(state["scene"].minimizer.computeNumericValue())


# ------------------------------------------------------------------------------ the least work


def _cube_counts(n):
    """(tets, moving vertices, upper 3x3 blocks) of the bottom-fixed cube."""
    m, layers = n + 1, n                        # moving vertices: m x m x layers
    axis = 2 * n * m * layers + m * m * (layers - 1)
    face = n * n * layers + 2 * n * m * (layers - 1)
    body = n * n * (layers - 1)
    return 6 * n ** 3, m * m * layers, m * m * layers + axis + face + body


def _assembly_work(tets, nv, nb, projected=0.6):
    # connectivity, rest shapes and positions in; gradient and blocks out
    return tets * (16 + 80) + nv * (24 + 24) + nb * 72, tets * (3000 + projected * 12000)


def _iterations(n, tol, solver):
    full = 2.25 * n * math.log(1.0 / tol) / math.log(1e6)
    return max(8.0, full * (0.55 if solver == "mas" else 1.0))


def work(case):
    kind = case["kind"]
    if kind in ("newton", "assembly", "spmv"):
        tets, nv, nb = _cube_counts(case["n"])
        a_bytes, a_flops = _assembly_work(tets, nv, nb, 0.0 if case.get("projection") == 0 else 0.6)
        if kind == "assembly":
            return {"bytes": a_bytes, "flops": a_flops}
        value = 36 if case.get("precision") == "mixed" else 72
        # blocks and their columns once, x and y
        product = nb * (value + 4) + 2 * 24 * nv
        if kind == "spmv":
            return {"bytes": product, "flops": 36.0 * nb}
        its = _iterations(case["n"], case["tol"], case["solver"])
        # per iteration: one product, the preconditioner, x, r, z, p, q in and out
        return {"bytes": a_bytes + its * (product + nv * (72 + 8 * 24)),
                "flops": a_flops + its * (36.0 * nb + 60.0 * nv)}
    if kind == "cloth":
        m = case["m"]
        tri, hinges, nv = 2 * (m - 1) ** 2, (m - 1) * (3 * m - 5) + 0, m * m
        nb = 7 * nv
        return {"bytes": tri * (12 + 40) + hinges * (16 + 16) + nv * 48 + nb * 72,
                "flops": tri * 3000.0 + hinges * 15000.0}
    if kind in ("contact", "ccd"):
        nb = case["bodies_x"] * case["bodies_z"]
        body_v = 0.6 * (case["cells"] + 1) ** 3
        cloth_v = case["cloth_m"] ** 2
        if kind == "ccd":
            prim = 5 * (cloth_v + nb * 6 * case["cells"] ** 2)
            return {"bytes": prim * 200.0, "flops": prim * 2000.0}
        blocks = 7 * (cloth_v + nb * body_v) + 6 * case["pairs"]
        its = 400.0
        return {"bytes": case["pairs"] * 300.0 + its * blocks * 76.0,
                "flops": case["pairs"] * 20000.0 + its * blocks * 36.0}
    if kind == "adjoint":
        tets, nv, nb = _cube_counts(case["n"])
        a_bytes, a_flops = _assembly_work(tets, nv, nb, 0.0)
        its = 8.0 * case["n"]
        return {"bytes": a_bytes + tets * 120 + its * (nb * 76 + nv * 300),
                "flops": a_flops + tets * 500.0 + its * 36.0 * nb}
    total = {"bytes": 0.0, "flops": 0.0}
    mean = math.sqrt(case["n_min"] * case["n_max"])
    for _ in range(case["count"]):
        w = work({"kind": "newton", "n": int(mean), "solver": "jacobian", "precision": "fp64",
                  "tol": 1e-6, "young": 1e5})
        total = {k: total[k] + w[k] for k in total}
    return total


# ------------------------------------------------------------------------------ tolerances


def tolerance(case):
    kind = case["kind"]
    if kind in ("newton", "serving"):
        # a solve stops at a residual of tol: the step is that residual times the operator's
        # inverse away from the exact one (six times tol at n = 48)
        return {"rel": 40.0 * case.get("tol", 1e-6), "max": 2000.0 * case.get("tol", 1e-6)}
    if kind == "contact":
        return {"rel": 1e-2, "max": 0.9}        # stiff barriers: the same, a thousand times
    if kind == "adjoint":
        return {"rel": 1e-7, "max": 1e-5}
    if kind == "ccd":
        return {"rel": 1e-12, "max": 1e-12}
    return {"rel": 1e-11, "max": 1e-9}          # FP64 sums and projections


# ------------------------------------------------------------------------------ in 64 bits


def _projected(H, method):
    """Symmetric matrices with their eigenvalues clamped (2) or turned positive (1)."""
    if method == 0:
        return H
    def part(A):
        w, V = np.linalg.eigh(A)
        w = np.abs(w) if method == 1 else np.maximum(w, 0.0)
        return (V * w[:, None, :]) @ np.swapaxes(V, 1, 2)
    parts = np.array_split(H, max(1, H.shape[0] // 20000))
    with ThreadPoolExecutor(min(16, os.cpu_count() or 1)) as pool:
        return np.concatenate(list(pool.map(part, parts)))


def _snh(x, rest, mu, lam, dt, method):
    """Gradients [T, 12] and Hessians [T, 12, 12] of Stable Neo-Hookean tets."""
    T = x.shape[0]
    Dm = np.stack([rest[:, k] - rest[:, 0] for k in (1, 2, 3)], 2)
    Di = np.linalg.inv(Dm)
    s = dt * dt * np.linalg.det(Dm) / 6.0
    Ds = np.stack([x[:, k] - x[:, 0] for k in (1, 2, 3)], 2)
    F = Ds @ Di
    cof = np.stack([np.cross(F[:, :, 1], F[:, :, 2]), np.cross(F[:, :, 2], F[:, :, 0]),
                    np.cross(F[:, :, 0], F[:, :, 1])], 2)
    ic = (F * F).sum((1, 2))
    J = (F[:, :, 0] * cof[:, :, 0]).sum(1)
    a1, a2 = mu * (1.0 - 1.0 / (ic + 1.0)), 2.0 * mu / (ic + 1.0) ** 2
    a3 = lam * (J - 1.0 - 0.75 * mu / lam)
    g = np.concatenate([-Di.sum(1, keepdims=True), Di], 1)            # [T, 4, 3]
    u, w = np.einsum("tij,taj->tai", F, g), np.einsum("tij,taj->tai", cof, g)
    grad = (s[:, None, None] * (a1[:, None, None] * u + a3[:, None, None] * w)).reshape(T, 12)
    H = np.empty((T, 4, 3, 4, 3))
    for a in range(4):
        for b in range(4):
            t = np.einsum("tij,tj->ti", F, np.cross(g[:, a], g[:, b]))
            B = a2[:, None, None] * u[:, a, :, None] * u[:, b, None, :] \
                + lam * w[:, a, :, None] * w[:, b, None, :]
            d = a1 * (g[:, a] * g[:, b]).sum(1)
            for i in range(3):
                B[:, i, i] += d
            for i, j, k, sign in ((0, 1, 2, -1), (1, 0, 2, 1), (0, 2, 1, 1), (2, 0, 1, -1),
                                  (1, 2, 0, -1), (2, 1, 0, 1)):
                B[:, i, j] -= sign * a3 * t[:, k]
            H[:, a, :, b, :] = s[:, None, None] * B
    return grad, _projected(H.reshape(T, 12, 12), method)


class _Blocks:
    """Gradient and upper 3x3 blocks, sorted by (row, column), from element terms."""

    def __init__(self, nv):
        self.nv, self.g, self.keys, self.vals = nv, np.zeros((nv, 3)), [], []

    def add(self, ids, grad, H):
        """ids [E, k] vertices (negative: fixed), grad [E, 3k], H [E, 3k, 3k]."""
        k = ids.shape[1]
        for a in range(k):
            ok = ids[:, a] >= 0
            for c in range(3):
                self.g[:, c] += np.bincount(ids[ok, a], grad[ok, 3 * a + c], self.nv)
            for b in range(k):
                up = ok & (ids[:, b] >= ids[:, a])
                self.keys.append(ids[up, a].astype(np.int64) * self.nv + ids[up, b])
                self.vals.append(H[up, 3 * a:3 * a + 3, 3 * b:3 * b + 3].reshape(-1, 9))

    def done(self):
        keys, inv = np.unique(np.concatenate(self.keys), return_inverse=True)
        vals = np.concatenate(self.vals)
        out = np.stack([np.bincount(inv, vals[:, j], keys.size) for j in range(9)], 1)
        return self.g.reshape(-1), keys // self.nv, keys % self.nv, out


def _cube_exact(case, seed, method):
    cs = _cube_case(case, seed)
    out = _Blocks(cs.n_moving)
    grad, H = _snh(cs.position[cs.tets], cs.rest[cs.tets], cs.mu, cs.lam, cs.dt, method)
    out.add(cs.tets - cs.n_fixed, grad, H)
    target = cs.last_position + cs.velocity * cs.dt - [0.0, 9.8 * cs.dt ** 2, 0.0]
    m = cs.mass[cs.n_fixed:, None]
    out.add(np.arange(cs.n_moving)[:, None], m * (cs.position - target)[cs.n_fixed:],
            m[:, :, None] * np.eye(3))
    return out.done()


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _product(rows, cols, vals, nv):
    """x -> A x of the symmetric matrix in upper blocks, in torch."""
    dev = _device()
    r, c = torch.from_numpy(rows).to(dev), torch.from_numpy(cols).to(dev)
    B = torch.from_numpy(vals).to(dev).reshape(-1, 3, 3)
    off = torch.nonzero(r != c).reshape(-1)
    ro, co, Bt = r[off], c[off], B[off].transpose(1, 2).contiguous()

    def apply(x):
        x = x.reshape(nv, 3)
        y = torch.zeros_like(x)
        y.index_add_(0, r, (B * x[c][:, None, :]).sum(2))
        y.index_add_(0, co, (Bt * x[ro][:, None, :]).sum(2))
        return y.reshape(-1)
    diag = torch.zeros(nv, 3, 3, dtype=torch.float64, device=dev)
    diag[r[r == c]] = B[r == c]
    return apply, diag


def _solve(rows, cols, vals, g):
    """A^-1 g to the rounding of 64 bits (conjugate gradients to 1e-13)."""
    nv = g.size // 3
    A, diag = _product(rows, cols, vals, nv)
    inv = torch.linalg.inv(diag.cpu()).to(diag.device)
    b = torch.from_numpy(g).to(diag.device)
    x, r = torch.zeros_like(b), b.clone()
    M = lambda v: (inv * v.reshape(nv, 1, 3)).sum(2).reshape(-1)      # noqa: E731
    z = M(r)
    p, rz = z.clone(), r @ z
    stop = 1e-13 * float(b.norm())
    for it in range(6000):
        q = A(p)
        alpha = rz / (p @ q)
        x += alpha * p
        r -= alpha * q
        if it % 8 == 0 and float(r.norm()) <= stop:
            break
        z = M(r)
        new = r @ z
        p = z + (new / rz) * p
        rz = new
    return x.cpu().numpy()


def _cloth_exact(case, seed):
    rest, tri, hinges = _cloth_mesh(case["m"])
    x = _cloth_positions(case["m"], seed)
    c = _CLOTH
    r = torch.from_numpy(rest)

    def minv(t):
        e1, e2 = r[t[:, 1]] - r[t[:, 0]], r[t[:, 2]] - r[t[:, 0]]
        n = torch.linalg.cross(e1, e2)
        u = e1 / e1.norm(dim=1, keepdim=True)
        v = torch.linalg.cross(n / n.norm(dim=1, keepdim=True), u)
        M = torch.stack([torch.stack([(u * e1).sum(1), (u * e2).sum(1)], 1),
                         torch.stack([(v * e1).sum(1), (v * e2).sum(1)], 1)], 1)
        return torch.linalg.inv(M), 0.5 * n.norm(dim=1) * c["thickness"]

    def stvk(y, Mi, vol):
        y = y.reshape(3, 3)
        F = torch.stack([y[1] - y[0], y[2] - y[0]], 1) @ Mi
        E = 0.5 * (F.transpose(0, 1) @ F - torch.eye(2, dtype=torch.float64))
        tr = E[0, 0] + E[1, 1]
        return vol * c["dt"] ** 2 * (c["mu"] * (E * E).sum() + 0.5 * c["lam"] * tr * tr)

    def angle(y):
        y = y.reshape(4, 3)
        cr = torch.linalg.cross
        n0, n1, a = cr(y[0] - y[2], y[1] - y[2]), cr(y[1] - y[3], y[0] - y[3]), y[1] - y[0]
        return 2.0 * torch.atan2((cr(n0, n1) @ a) / a.norm(), n0 @ n1 + n0.norm() * n1.norm())

    def bending(y, t0, length):
        return c["bend"] * (angle(y) - t0) ** 2 * length

    out = _Blocks(x.shape[0])
    X = torch.from_numpy(x)
    th = torch.from_numpy(hinges)
    rest_angle = torch.func.vmap(angle)(r[th].reshape(-1, 12))
    length = (r[th[:, 1]] - r[th[:, 0]]).norm(dim=1)
    for conn, f, args in ((tri, stvk, minv(torch.from_numpy(tri))),
                          (hinges, bending, (rest_angle, length))):
        y = X[torch.from_numpy(conn)].reshape(conn.shape[0], -1)
        grad = torch.func.vmap(torch.func.grad(f))(y, *args).numpy()
        H = torch.func.vmap(torch.func.hessian(f))(y, *args).numpy()
        out.add(conn, grad, _projected(0.5 * (H + np.swapaxes(H, 1, 2)), case["projection"]))
    return out.done()


def exact(case, seed):
    kind = case["kind"]
    if kind in ("newton", "assembly", "spmv"):
        if case["n"] > 50:
            return None                         # over 20 seconds
        g, rows, cols, vals = _cube_exact(case, seed, case.get("projection", 2))
        out = {"gradient": g, "hessian": vals.reshape(-1)}
        if kind == "spmv":
            A, _ = _product(rows, cols, vals, g.size // 3)
            return {"y": A(torch.from_numpy(_spmv_vector(g.size, seed)).to(_device())).cpu().numpy()}
        if kind == "newton":
            out["step"] = [_solve(rows, cols, vals, g)]
        return out
    if kind == "cloth":
        g, _, _, vals = _cloth_exact(case, seed)
        return {"gradient": g, "hessian": vals.reshape(-1)}
    if kind == "serving":
        from yasps_amd.serving import request_positions, serving_stream
        out = []
        fixed = serving_stream(case["count"], case["n_min"], case["n_max"], seed=7)
        for a, b in zip(serving_stream(case["count"], case["n_min"], case["n_max"], seed=seed), fixed):
            a.n = b.n
            from yasps_amd.scenes import lame_parameters
            base = _cube(a.n)
            x = base.rest.copy()
            x[base.n_fixed:] = request_positions(base, a)
            mu, lam = lame_parameters(a.young, base.poisson)
            blocks = _Blocks(base.n_moving)
            grad, H = _snh(x[base.tets], base.rest[base.tets], mu, lam, base.dt, 2)
            blocks.add(base.tets - base.n_fixed, grad, H)
            target = base.last_position - [0.0, 9.8 * base.dt ** 2, 0.0]
            m = base.mass[base.n_fixed:, None]
            blocks.add(np.arange(base.n_moving)[:, None], m * (x - target)[base.n_fixed:],
                       m[:, :, None] * np.eye(3))
            g, rows, cols, vals = blocks.done()
            out.append(_solve(rows, cols, vals, g))
        return out
    return None
