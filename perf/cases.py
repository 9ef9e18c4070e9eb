"""The work that a user of udx gives it, as cases to time: solvent boxes from
the smallest to the headline channel, the one-call-per-module binding, the
ensemble, red-cell suspensions and the membrane forces with their adjoint.

A case is a dict of plain values; prepare() makes what a simulation program
holds before the call (particles made from a seed, the solver's handles) and
run() is one pass of such a program: a few steps and the particles and forces
read back, or one force evaluation.  Simulations carry on from pass to pass.
"""
import math

import numpy as np
import torch

from ctc_amd import udx as U

DT, KBT = 5e-4, 0.0444

# rbc.test.cfg: the membrane coefficients of the reference's tests
RBC = dict(gammaC=30.0, gammaT=90.0, kBT=0.0444, kb=17.78, phi=6.97, ks=14.8, x0=0.5, mpow=2.0, ka=2450.0,
           kd=100.0, kv=3750.0)


def listed():
    return [
        # the 16^3 test box of bench.py: 12 thousand particles, step pairs replayed from a graph;
        # what a parameter scan of small boxes runs, bound by latency
        {"name": "box16", "kind": "box", "Lx": 16, "Ly": 16, "Lz": 16, "rho": 3, "a": 75.0, "g": 4.5, "kBT": 1.0,
         "dt": 1e-3, "spow": 0.25, "steps": 10, "graph": True, "half": False},
        # a small ragged box, launched step by step
        {"name": "box_ragged", "kind": "box", "Lx": 31, "Ly": 17, "Lz": 24, "rho": 5, "a": 25.0, "g": 6.0, "kBT": 0.5,
         "dt": 1e-3, "spow": 0.5, "steps": 4, "graph": False, "half": False},
        # an ordinary box at the blood-plasma density of the reference's configuration
        {"name": "box48", "kind": "box", "Lx": 48, "Ly": 48, "Lz": 48, "rho": 10, "a": 2.6666667, "g": 8.0,
         "kBT": KBT, "dt": DT, "spow": 0.25, "steps": 1, "graph": False, "half": False},
        # the force mode with order-independent sums
        {"name": "box_half_shell", "kind": "box", "Lx": 40, "Ly": 36, "Lz": 44, "rho": 8, "a": 2.6666667, "g": 8.0,
         "kBT": KBT, "dt": DT, "spow": 0.25, "steps": 1, "graph": False, "half": True},
        # bench.py's headline: Poiseuille flow between plane walls, 7.4 million solvent particles
        {"name": "channel96", "kind": "channel", "Lx": 96, "Ly": 96, "Lz": 96, "rho": 10, "h": 40.0, "gdot": 0.0,
         "grid": 128, "steps": 4},
        # a small Couette cell: shearing walls, an odd side
        {"name": "couette_small", "kind": "channel", "Lx": 33, "Ly": 24, "Lz": 28, "rho": 6, "h": 10.0, "gdot": 0.05,
         "grid": 48, "steps": 4},
        # a program with its own loop that binds module by module: cell list, then forces on AoS arrays
        {"name": "forces_binding", "kind": "forces", "Lx": 40, "Ly": 33, "Lz": 37, "rho": 4, "a": 50.0, "g": 4.5,
         "kBT": 1.0, "dt": 1e-3, "spow": 0.25},
        # bench.py's ensemble: uneven boxes advanced together
        {"name": "ensemble64", "kind": "ensemble", "boxes": 64, "lo": 8, "hi": 48, "pick": 2024, "steps": 4},
        # bench.py's suspension at hematocrit 0.2: 512 red cells in a 64^3 box
        {"name": "suspension64", "kind": "suspension", "nx": 8, "ny": 8, "nz": 8, "rho": 10, "sub": 3, "walls": False,
         "steps": 2},
        # a few red cells between shearing walls, with contact and wall repulsion
        {"name": "cells_in_channel", "kind": "suspension", "nx": 4, "ny": 4, "nz": 2, "rho": 10, "sub": 2,
         "walls": True, "steps": 2},
        # calibration of the membrane coefficients: force and adjoint of 256 cells (bench.py's adjoint leg)
        {"name": "membranes256", "kind": "membranes", "cells": 256, "sub": 3, "adjoint": True},
        # the stretch test of one cell: force, point loads, vertex kick-drift
        {"name": "one_cell_stretch", "kind": "membranes", "cells": 1, "sub": 3, "adjoint": False},
    ]


def draw(rng):
    def logint(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    dpd = {"a": rng.choice([2.6666667, 25.0, 75.0]), "g": round(rng.uniform(4.0, 10.0), 3),
           "kBT": round(rng.uniform(0.04, 1.0), 3), "dt": rng.choice([5e-4, 1e-3]), "spow": rng.choice([0.25, 0.25, 0.5])}
    kind = rng.choice(["box", "box", "box", "forces", "channel", "channel", "ensemble", "suspension", "suspension",
                       "membranes"])
    if kind == "box":
        L, rho = [logint(12, 72) for _ in range(3)], rng.randint(3, 10)
        return dict({"kind": kind, "Lx": L[0], "Ly": L[1], "Lz": L[2], "rho": rho,
                     "steps": 4 if rho * L[0] * L[1] * L[2] < 60_000 else 1, "graph": rng.random() < 0.5,
                     "half": rng.random() < 0.2}, **dpd)
    if kind == "forces":
        return dict({"kind": kind, "Lx": logint(12, 64), "Ly": logint(12, 64), "Lz": logint(12, 64),
                     "rho": rng.randint(3, 10)}, **dpd)
    if kind == "channel":
        Lz = 2 * logint(12, 42)
        return {"kind": kind, "Lx": logint(16, 84), "Ly": logint(16, 84), "Lz": Lz, "rho": rng.randint(4, 10),
                "h": 0.5 * Lz - rng.choice([3.0, 4.0, 6.0]), "gdot": rng.choice([0.0, 0.05]), "grid": 64, "steps": 4}
    if kind == "ensemble":
        return {"kind": kind, "boxes": logint(4, 56), "lo": 8, "hi": rng.randint(16, 48),
                "pick": rng.randint(0, 10 ** 6), "steps": 4}
    if kind == "suspension":
        walls = rng.random() < 0.4
        return {"kind": kind, "nx": rng.randint(2, 7), "ny": rng.randint(2, 7), "nz": rng.randint(1 if walls else 2, 7),
                "rho": rng.randint(6, 10), "sub": rng.choice([2, 3]), "walls": walls, "steps": 2}
    return {"kind": kind, "cells": logint(1, 256), "sub": rng.choice([2, 3]), "adjoint": rng.random() < 0.6}


# ---------------------------------------------------------------- inputs
def gen_of(seed, *salt):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + sum((k + 1) * 7919 * int(s) for k, s in enumerate(salt))) % (1 << 62))
    return g


def fluid(L, rho, kBT, g):
    """rho particles in every unit cell, uniform inside it (the reference's
    initial condition), Maxwell velocities without net momentum"""
    nc = L[0] * L[1] * L[2]
    c = torch.arange(nc, device="cuda").repeat_interleave(rho)
    org = torch.stack([c % L[0], c // L[0] % L[1], c // (L[0] * L[1])], 1).double()
    half = torch.tensor([0.5 * x for x in L], device="cuda", dtype=torch.float64)
    r = org + torch.rand((nc * rho, 3), generator=g, device="cuda") * (1 - 1e-5) - half
    v = torch.randn((nc * rho, 3), generator=g, device="cuda", dtype=torch.float64) * math.sqrt(kBT)
    pp = torch.cat([r, v - v.mean(0)], 1).float()
    return pp[torch.randperm(len(pp), generator=g, device="cuda")].contiguous()


def red_cell(sub, diameter):
    """biconcave red cell: an icosahedron subdivided `sub` times (162 vertices
    for 2, 642 for 3) mapped by Evans' and Fung's profile"""
    t = (1 + 5 ** 0.5) / 2
    v = [[-1, t, 0], [1, t, 0], [-1, -t, 0], [1, -t, 0], [0, -1, t], [0, 1, t], [0, -1, -t], [0, 1, -t], [t, 0, -1],
         [t, 0, 1], [-t, 0, -1], [-t, 0, 1]]
    f = [[0, 11, 5], [0, 5, 1], [0, 1, 7], [0, 7, 10], [0, 10, 11], [1, 5, 9], [5, 11, 4], [11, 10, 2], [10, 7, 6],
         [7, 1, 8], [3, 9, 4], [3, 4, 2], [3, 2, 6], [3, 6, 8], [3, 8, 9], [4, 9, 5], [2, 4, 11], [6, 2, 10],
         [8, 6, 7], [9, 8, 1]]
    v = [np.array(x, float) / math.sqrt(1 + t * t) for x in v]
    for _ in range(sub):
        mid, nf = {}, []
        for a, b, c in f:
            m = []
            for i, j in ((a, b), (b, c), (c, a)):
                k = (min(i, j), max(i, j))
                if k not in mid:
                    x = v[i] + v[j]
                    mid[k] = len(v)
                    v.append(x / np.linalg.norm(x))
                m.append(mid[k])
            nf += [[a, m[0], m[2]], [b, m[1], m[0]], [c, m[2], m[1]], m]
        f = nf
    v = np.array(v)
    q = v[:, 0] ** 2 + v[:, 1] ** 2
    v[:, 2] *= 0.5 * (0.2072 + 2.0026 * q - 1.1228 * q * q)
    return (v * (0.5 * diameter)).astype(np.float32), np.array(f, np.int32)


def mesh_size(rr, tt):
    a, b, c = (rr[tt[:, k]].astype(np.float64) for k in range(3))
    return 0.5 * np.linalg.norm(np.cross(b - a, c - a), axis=1).sum(), (a * np.cross(b, c)).sum() / 6.0


def turned(rr, centres, g):
    """copies of the template in random orientations at the centres"""
    n = len(centres)
    q = torch.nn.functional.normalize(torch.randn((n, 4), generator=g, device="cuda", dtype=torch.float64), dim=1)
    w, x, y, z = q.unbind(1)
    R = torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                     2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                     2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], 1).reshape(n, 3, 3)
    r = torch.as_tensor(rr, device="cuda", dtype=torch.float64)
    out = (R[:, None] * r[None, :, None, :]).sum(-1) + torch.as_tensor(centres, device="cuda")[:, None]
    return out.reshape(-1, 3)


class State(dict):
    """what the program holds; its handles are closed with it, the last made first"""

    def __del__(self):
        try:
            for h in reversed(self.get("handles", [])):
                h.close()
        except Exception:
            pass


def channel_walls(st, ctx, L, h, grid, gdot, pp):
    """plane channel |z| < h: the walls frozen from the fluid; returns the solvent that stays"""
    z = (np.arange(grid) + 0.5) * (L[2] / grid) - 0.5 * L[2]
    D = np.ascontiguousarray(np.broadcast_to((np.abs(z) - h).astype(np.float32)[:, None, None], (grid,) * 3))
    sdf = U.Sdf(ctx, L, ext=[float(x) for x in L], N=(grid,) * 3, D=D)
    wall = U.Wall(ctx, sdf, pp)
    st["handles"] += [sdf, wall]
    if gdot:
        wall.set_vel(U.wall_vel("shear", gdot=gdot, vdir=0, gdir=2))
    # the fluid's cells end at the walls: all but a few particles' worth of rounding are known to stay
    n = min(wall.n_solvent, len(pp) // L[2] * int(round(2 * h)) - 64)
    return wall, pp[:n].contiguous()


def ensemble_boxes(case):
    rng = np.random.default_rng(case["pick"])
    out = []
    for _ in range(case["boxes"]):
        L = tuple(int(x) for x in rng.integers(case["lo"], case["hi"] + 1, 3))
        out.append(dict(L=L, rho=int(rng.choice([3, 5, 10])), g=float(rng.uniform(4, 10)),
                        kBT=float(rng.uniform(0.04, 1.0))))
    return out


def box_size(case):
    return (case["Lx"], case["Ly"], case["Lz"])


def suspension_size(case):
    """one red cell of diameter 7.8 per 8 x 8 x 8 block (8 x 8 x 9 between walls)"""
    L = (8 * case["nx"], 8 * case["ny"], 8 * case["nz"])
    return L if not case["walls"] else (L[0], L[1], 2 * ((9 * case["nz"] + 1) // 2) + 8)


def prepare(case, seed):
    kind, ctx = case["kind"], U.Context()
    st = State(handles=[ctx], kind=kind)
    g = gen_of(seed, 1)
    if kind == "box":
        L = box_size(case)
        pp = fluid(L, case["rho"], case["kBT"], g)
        par = U.dpd_params(case["a"], case["g"], case["kBT"], case["dt"], case["spow"])
        flu = U.Flu(ctx, L, len(pp), par, case["dt"], mode=U.MODE_HALF if case["half"] else U.MODE_FAST)
        flu.set_pp(pp)
        if case["graph"]:
            flu.graph(True)
    elif kind == "channel":
        L = box_size(case)
        wall, pp = channel_walls(st, ctx, L, case["h"], case["grid"], case["gdot"], fluid(L, case["rho"], KBT, g))
        flu = U.Flu(ctx, L, len(pp), U.dpd_params(2.5, 8.0, KBT, DT, 0.25), DT, 1.0, (0.01, 0.0, 0.0))
        flu.set_pp(pp)
        flu.set_wall(wall)
    elif kind == "forces":
        L = box_size(case)
        pp = fluid(L, case["rho"], case["kBT"], g)
        st.update(pp=pp, out=torch.empty_like(pp), ff=torch.empty((len(pp), 3), device="cuda"),
                  par=U.dpd_params(case["a"], case["g"], case["kBT"], case["dt"], case["spow"]),
                  seeds=np.random.default_rng(seed).random(27).astype(np.float32),
                  cl=U.Clist(ctx, L, len(pp)), flu=U.FluForces(ctx, L, len(pp)))
        st["handles"] += [st["cl"], st["flu"]]
        return st
    elif kind == "ensemble":
        boxes, pps = [], []
        for k, b in enumerate(ensemble_boxes(case)):
            pp = fluid(b["L"], b["rho"], b["kBT"], gen_of(seed, 1, k))
            boxes.append(dict(L=b["L"], n=len(pp), params=U.dpd_params(25.0, b["g"], b["kBT"], 1e-3, 0.25), dt=1e-3))
            pps.append(pp)
        pp = torch.cat(pps)
        ens = U.Ensemble(ctx, boxes)
        ens.set_pp(pp)
        ens.graph(True)
        st["handles"].append(ens)
        st.update(ens=ens, steps=case["steps"], pp=torch.empty_like(pp))
        return st
    elif kind == "suspension":
        L = suspension_size(case)
        pp, wall = fluid(L, case["rho"], KBT, g), None
        h = 0.5 * L[2] - 4.0
        if case["walls"]:
            wall, pp = channel_walls(st, ctx, L, h, 64, 0.05, pp)
        rr, tt = red_cell(case["sub"], 7.8)
        n = (case["nx"], case["ny"], case["nz"])
        sp = (8.0, 8.0, 2 * h / n[2] if wall else 8.0)
        grid = np.stack(np.meshgrid(*[(np.arange(n[c]) + 0.5 - 0.5 * n[c]) * sp[c] for c in range(3)], indexing="ij"), -1)
        x = turned(rr, grid.reshape(-1, 3), g)
        vert = torch.cat([x, torch.randn(x.shape, generator=g, device="cuda", dtype=torch.float64) * 0.05], 1).float()
        nc = n[0] * n[1] * n[2]
        A, V = mesh_size(rr, tt)
        pair = U.dpd_params(2.6666667, 8.0, KBT, DT, 0.25)
        flu = U.Flu(ctx, L, len(pp), pair, DT, 1.0, (0.01, 0.0, 0.0) if wall else (0.0, 0.0, 0.0))
        flu.set_pp(pp)
        rbc = U.Rbc(ctx, tt, len(rr), nc)
        rbc.set_stressfree(rr)
        fsi = U.Fsi(ctx, L, nc * len(rr))
        flu.set_rbc(rbc, fsi, U.rbc_params(totArea=A, totVolume=V, **dict(RBC, kb=40.0)), pair, 0.5, 1, nc, vert)
        st["handles"] += [rbc, fsi]
        if wall:
            cnt = U.Cnt(ctx, L, nc * len(rr))
            flu.set_wall(wall)
            flu.set_rbc_repulsion(2.0)
            flu.set_rbc_contact(cnt, U.PairDpdLj(2.6666667, 8.0, pair.s, 0.25, 0.3, 0.44))
            st["handles"].append(cnt)
        st["vert"] = vert
    else:
        rr, tt = red_cell(case["sub"], 6.0)
        nc, nv = case["cells"], len(rr)
        k = np.arange(nc)
        x = turned(rr, np.stack([12.0 * (k % 16), 12.0 * (k // 16), 0.0 * k], 1), g)
        x = x + torch.randn(x.shape, generator=g, device="cuda", dtype=torch.float64) * 0.02
        u = torch.randn(x.shape, generator=g, device="cuda", dtype=torch.float64) * (0.0 if case["adjoint"] else 0.05)
        A, V = mesh_size(rr, tt)
        rbc = U.Rbc(ctx, tt, nv, nc)
        rbc.set_stressfree(rr)
        coef = dict(RBC, gammaC=0.0, gammaT=0.0) if case["adjoint"] else RBC
        st.update(ctx=ctx, rbc=rbc, par=U.rbc_params(totArea=A, totVolume=V, **coef), cells=nc, nv=nv,
                  adjoint=case["adjoint"], pp0=torch.cat([x, u], 1).float(),
                  ff=torch.empty((nc * nv, 3), device="cuda"), load=stretch_load(rr))
        st["handles"].append(rbc)
        if case["adjoint"]:
            st.update(g=torch.randn((nc * nv, 3), generator=g, device="cuda"), gx=torch.empty_like(st["ff"]))
        else:
            st["pp"] = torch.empty_like(st["pp0"])
        return st
    st["handles"].append(flu)
    st.update(flu=flu, steps=case["steps"], pp=torch.empty_like(pp), ff=torch.empty((len(pp), 3), device="cuda"))
    return st


def stretch_load(rr):
    """opposed loads along x on the 5% of vertices at the two ends"""
    load, order, n = np.zeros((len(rr), 3), np.float32), np.argsort(rr[:, 0]), max(1, len(rr) // 40)
    load[order[:n], 0] = -7.0 / n
    load[order[-n:], 0] = 7.0 / n
    return torch.as_tensor(load).cuda()


# ---------------------------------------------------------------- one pass
def run(st):
    kind = st["kind"]
    if kind == "forces":
        n = st["cl"].build(st["pp"], st["out"])
        st["ff"].zero_()
        st["flu"].prepare(st["out"][:n])
        st["flu"].apply(st["par"], st["cl"].starts_ptr(), st["ff"], seeds=st["seeds"])
        return st["out"], st["ff"]
    if kind == "ensemble":
        st["ens"].run(st["steps"])
        st["ens"].get_pp(st["pp"])
        return st["pp"]
    if kind == "membranes":
        st["ff"].zero_()
        if st["adjoint"]:
            st["rbc"].force(st["par"], 0.0, st["cells"], st["pp0"], st["ff"])
            return st["ff"], st["gx"], st["rbc"].adjoint(st["par"], st["cells"], st["pp0"], st["g"], st["gx"])
        st["pp"].copy_(st["pp0"])
        st["rbc"].force(st["par"], DT, st["cells"], st["pp"], st["ff"])
        U.rbc_stretch_apply(st["ctx"], st["cells"], st["nv"], st["load"], st["ff"])
        U.scheme_move_apply(st["ctx"], DT, 0.5, st["ff"], st["pp"])
        return st["ff"], st["pp"]
    st["flu"].run(st["steps"])
    st["flu"].get_pp(st["pp"])
    st["flu"].get_ff(st["ff"])
    return (st["pp"], st["ff"]) if kind != "suspension" else (st["pp"], st["ff"], st["vert"])


def work(case):
    """bytes: per step the particles read once and written once, per pass the
    particles and forces read back; flops: 100 per interacting pair (once per
    pair) and 9 per half-shell distance test, 1200 (FP64) per ring slot of a
    membrane vertex and three times that for its adjoint"""
    def solvent(n, rho, steps):
        pairs = n * rho * 2.0 * math.pi / 3.0
        return n * (48.0 * steps + 60.0), steps * (pairs * 100.0 + n * 13.5 * rho * 9.0)

    kind = case["kind"]
    if kind == "membranes":
        n = case["cells"] * (10 * 4 ** case["sub"] + 2)
        a = 3 if case["adjoint"] else 0
        return {"bytes": n * (24.0 + 12.0 + (48.0 if a else 24.0)), "flops": n * 6 * 1200.0 * (1 + a)}
    if kind == "ensemble":
        w = [solvent(b["rho"] * b["L"][0] * b["L"][1] * b["L"][2], b["rho"], case["steps"])
             for b in ensemble_boxes(case)]
        return {"bytes": sum(x[0] for x in w), "flops": sum(x[1] for x in w)}
    L = suspension_size(case) if kind == "suspension" else box_size(case)
    n = float(case["rho"] * L[0] * L[1] * L[2])
    if kind == "forces":
        b, f = solvent(n, case["rho"], 1)
        return {"bytes": n * 60.0, "flops": f}
    if kind == "channel":
        n *= 2 * case["h"] / L[2]
    if kind == "suspension" and case["walls"]:
        n *= (L[2] - 8.0) / L[2]
    b, f = solvent(n, case["rho"], case["steps"])
    if kind == "suspension":
        nv = case["nx"] * case["ny"] * case["nz"] * (10 * 4 ** case["sub"] + 2)
        pairs = nv * case["rho"] * 4.0 * math.pi / 3.0
        b += case["steps"] * nv * 72.0
        f += case["steps"] * (pairs * 100.0 + nv * (27.0 * case["rho"] * 9.0 + 6 * 1200.0))
    return {"bytes": b, "flops": f}


def tolerance(case):
    """about four times the distance from the 64-bit results seen over these
    ranges: one evaluation of the pair forces 1e-5 (a pair near the cutoff,
    where the weight (1 - r)^spow is steep), a few steps 5e-5, the membrane
    terms (FP64, stored in 32 bits) 7e-7 in the summed coefficient gradients"""
    if case["kind"] == "membranes":
        return {"rel": 3e-6}
    return {"rel": 5e-5 if case["kind"] == "forces" or case["steps"] == 1 else 2e-4}


# ---------------------------------------------------------------- 64 bits
GOLD, SILVER = np.float32(0.6180339887498948482), np.float32(0.4142135623730950488)
BRONZE, TIN = np.float32(0.00008877875787352212838853023), np.float32(0.00004602357186447026756768986)


def kiss(x, y, z, c):
    """the KISS generator's floats in [0, 1]"""
    M = 0xFFFFFFFF
    while True:
        x = (69069 * x + 12345) & M
        y ^= (y << 13) & M
        y ^= y >> 17
        y ^= (y << 5) & M
        t = 698769069 * z + c
        c, z = t >> 32, t & M
        yield float(np.float32((x + y + z) & M) / np.float32(M))


def trunks(offset=0):
    """the seed streams of the 26 halo fragments and the bulk"""
    out = []
    for f in range(26):
        d = ((f + 2) % 3 - 1, (f // 3 + 2) % 3 - 1, (f // 9 + 2) % 3 - 1)
        s = sum(d)
        plus = s > 0 or (s == 0 and d[0] > 0) or (d[0] == 0 and d[1] > 0) or (d[1] == 0 and d[2] > 0)
        v = [1 + (1 if plus else -1) * x for x in d]
        seed = v[0] + 3 * (v[1] + 3 * v[2])
        out.append(kiss((390 + seed + offset) & 0xFFFFFFFF, seed + 615, 12309, 23094))
    return out + [kiss(offset & 0xFFFFFFFF, 0, 0, 0)]


def noise(seed, u, v):
    """mean 0, variance 1 number of an index pair: a low-discrepancy point and
    18 logistic maps in 32 bits as defined (products rounded to nearest, the
    two fused steps toward zero), which any implementation has to give exactly"""
    def f32(x):
        return x.float().double()

    def down(x):   # toward zero to 24 bits
        return (x.view(torch.int64) & -(1 << 29)).view(torch.float64)

    u, v = u.double(), v.double()
    s = f32(f32(u) * float(BRONZE))
    s = f32(torch.remainder(u, 1024) * float(GOLD) + s)
    s = f32(torch.remainder(v, 1024) * float(SILVER) + s)
    s = f32(f32(v) * float(TIN) + s)
    x = f32(float(np.float32(seed)) - (s - torch.floor(s)))
    for _ in range(9):
        x2 = f32(x * x)
        x = down(down(8.0 * x2 - 8.0) * x2 + 1.0)
    return x * float(np.float32(1.41421356237309514547))


def dpd64(L, r, v, par, seeds, sub):
    """particles in cell order (stable; x slabs of 1/sub inside a cell) and
    their forces, pair by pair in 64 bits"""
    a, gamma, sigma, spow = par
    Lt = torch.tensor([float(x) for x in L], dtype=torch.float64, device=r.device)
    c = torch.floor(r + 0.5 * Lt).long()
    slab = torch.floor((r[:, 0] + 0.5 * L[0]) * sub).long() - c[:, 0] * sub
    cell = c[:, 0] + L[0] * (c[:, 1] + L[1] * c[:, 2])
    order = torch.argsort(cell * sub + slab, stable=True)
    r, v, c, cell = r[order], v[order], c[order], cell[order]
    n, nc = len(r), L[0] * L[1] * L[2]
    count = torch.bincount(cell, minlength=nc)
    start = torch.cumsum(count, 0) - count
    most = int(count.max())
    f = torch.zeros_like(r)
    lists = {}

    def place(d):   # position in the packed list of the boundary cells toward d
        if d not in lists:
            m = torch.ones(n, dtype=torch.bool, device=r.device)
            for k in range(3):
                if d[k]:
                    m &= c[:, k] == (L[k] - 1 if d[k] > 0 else 0)
            lists[d] = torch.cumsum(m, 0) - 1
        return lists[d]

    def fid(d):
        return (d[0] + 2) % 3 + 3 * ((d[1] + 2) % 3) + 9 * ((d[2] + 2) % 3)

    def add(i, j, w):
        dr = r[i] - torch.tensor([float(w[k] * L[k]) for k in range(3)], dtype=torch.float64, device=r.device) - r[j]
        r2 = (dr * dr).sum(1)
        ok = (r2 < 1.0) & ((i != j) if w == (0, 0, 0) else True)
        i, j, dr, r2 = i[ok], j[ok], dr[ok], r2[ok]
        if w == (0, 0, 0):
            rnd = noise(seeds[26], torch.maximum(i, j), torch.minimum(i, j))
        else:
            back = tuple(-x for x in w)
            p, q = place(w)[i], place(back)[j]
            rnd = noise(seeds[fid(w)], *((p, q) if fid(w) < fid(back) else (q, p)))
        far = r2 >= 1e-6
        d = torch.where(far, r2.sqrt(), torch.zeros_like(r2))
        e = torch.where(far[:, None], dr / torch.where(far, d, torch.ones_like(d))[:, None], torch.zeros_like(dr))
        rm = 1.0 - d
        wr = rm ** spow
        ev = (e * (v[i] - v[j])).sum(1)
        f.index_add_(0, i, ((-gamma * wr * ev + sigma * rnd) * wr + a * rm)[:, None] * e)

    every = torch.arange(n, device=r.device)
    for oz in (-1, 0, 1):
        for oy in (-1, 0, 1):
            for ox in (-1, 0, 1):
                q = c + torch.tensor([ox, oy, oz], device=r.device)
                w = torch.div(q, torch.tensor(L, device=r.device), rounding_mode="floor")
                q = q - w * torch.tensor(L, device=r.device)
                nb = q[:, 0] + L[0] * (q[:, 1] + L[1] * q[:, 2])
                code = (w[:, 0] + 1) + 3 * (w[:, 1] + 1) + 9 * (w[:, 2] + 1)
                for wc in torch.unique(code).tolist():
                    ww = (wc % 3 - 1, wc // 3 % 3 - 1, wc // 9 - 1)
                    mine = every[code == wc]
                    for k in range(most):
                        i = mine[count[nb[mine]] > k]
                        if len(i):
                            add(i, start[nb[i]] + k, ww)
    return r, v, f


def box64(L, pp, par, dt, steps, offset=0):
    """the box after `steps` steps of forces, kick-drift and periodic wrap"""
    r, v = pp[:, :3].double(), pp[:, 3:].double()
    Lt = torch.tensor([float(x) for x in L], dtype=torch.float64, device=r.device)
    tr = trunks(offset)
    for _ in range(steps):
        r, v, f = dpd64(L, r, v, par, [next(t) for t in tr], 4)
        v = v + f * float(np.float32(dt))
        r = r + v * float(np.float32(dt))
        r = torch.where(r < -0.5 * Lt, r + Lt, torch.where(r >= 0.5 * Lt, r - Lt, r))
    return torch.cat([r, v], 1), f


def par64(a, g, kBT, dt, spow):
    f = np.float32
    return (float(f(a)), float(f(g)), float(np.sqrt(f(2) * f(kBT) * f(g) / f(dt))), spow)


def membrane64(case, seed):
    """the ring walk of every vertex as tensor operations, and its derivative along the cotangent"""
    st = prepare(case, seed)
    rr, tt = red_cell(case["sub"], 6.0)
    nc, nv, dev = case["cells"], len(rr), "cuda"
    third = {}
    for a, b, c in tt.tolist():
        third[a, b], third[b, c], third[c, a] = c, a, b
    half = [(v, i1, i2, third[v, i2], third[i2, i1]) for (v, i1), i2 in third.items()]
    v, i1, i2, i3, i4 = (torch.tensor(h, device=dev) for h in zip(*half))
    p0 = torch.as_tensor(rr.astype(np.float64), device=dev)
    l0 = (p0[v] - p0[i1]).norm(dim=1).float().double()
    a0 = (0.5 * torch.linalg.cross(p0[i1] - p0[v], p0[i2] - p0[v]).norm(dim=1)).float().double()
    t = torch.as_tensor(tt.astype(np.int64), device=dev)
    P = {k: float(getattr(st["par"], k)) for k in ("ka", "kd", "kv", "ks", "x0", "mpow", "kb", "phi", "gammaC", "gammaT",
                                                   "totArea", "totVolume")}
    phi = P["phi"] / 180.0 * math.pi
    cross = torch.linalg.cross

    def dot(x, y):
        return (x * y).sum(-1, keepdim=True)

    def angle(a, b, c, d, first):
        ab, ac, cd, bd, bc, da = a - b, a - c, c - d, b - d, b - c, d - a
        k, n = cross(ab, ac), cross(bd, bc)
        ok, on = 1 / dot(k, k).sqrt(), 1 / dot(n, n).sqrt()
        cos = dot(k, n) * ok * on
        s2 = 1 - cos * cos
        sin = 1 / torch.where(s2 > 1e-6, s2, torch.full_like(s2, 1e-6)).sqrt()
        sin = torch.where(dot(k - n, da) < 0, -sin, sin)
        beta = math.cos(phi) - cos * math.sin(phi) * sin
        b11, b12, b22 = -beta * cos * ok * ok, beta * ok * on, -beta * cos * on * on
        if first:
            return b11 * cross(k, c - b) + b12 * cross(n, c - b)
        return b11 * cross(k, ac) + b12 * (cross(k, cd) + cross(n, ac)) + b22 * cross(n, cd)

    def terms(x):
        x = x.reshape(nc, nv, 3)
        q0, q1, q2 = x[:, t[:, 0]], x[:, t[:, 1]], x[:, t[:, 2]]
        area = 0.5 * cross(q1 - q0, q2 - q0).norm(dim=-1).sum(1)[:, None, None]
        vol = dot(q0, cross(q1, q2)).sum(1)[:, None] / 6
        r1, r2, r3 = x[:, v], x[:, i1], x[:, i2]
        nn = cross(r2 - r1, r3 - r1)
        f, a = cross(nn, r3 - r2), 0.5 * nn.norm(dim=-1, keepdim=True)
        lm, l = (l0 / P["x0"])[:, None], l0[:, None]

        def wlc(s):
            y = s / lm
            return (4 * y * y - 9 * y + 6) / (4 * (y - 1) * (y - 1)) / lm

        s = (r2 - r1).norm(dim=-1, keepdim=True)
        s = torch.where(s >= lm, 0.99 * lm.expand_as(s), s)
        m = P["mpow"] + 1
        out = [-(area - P["totArea"]) / (4 * P["totArea"] * a) * f, -(a - a0[:, None]) / (4 * a0[:, None] * a) * f,
               (vol - P["totVolume"]) / (6 * P["totVolume"]) * cross(r3, r2),
               (wlc(s) - wlc(l) * (l / s) ** m) * (r2 - r1),
               angle(r1, r3, r2, x[:, i4], True) + angle(r2, r1, r3, x[:, i3], False)]
        return [torch.zeros_like(x).index_add(1, v, o).reshape(-1, 3) for o in out]

    coef = [P[k] for k in ("ka", "kd", "kv", "ks", "kb")]
    pp = st["pp0"].double()
    x = pp[:, :3]
    F = sum(c * o for c, o in zip(coef, terms(x)))
    if case["adjoint"]:
        g = st["g"].double()
        out, gx = torch.func.jvp(lambda y: sum(c * o for c, o in zip(coef, terms(y))), (x,), (g,))
        return F, gx, [float((g * o).sum()) for o in terms(x)]
    xv, uv = x.reshape(nc, nv, 3), pp[:, 3:].reshape(nc, nv, 3)
    du, dr = uv[:, i1] - uv[:, v], xv[:, v] - xv[:, i1]
    visc = P["gammaT"] * du + P["gammaC"] * dot(du, dr) / dot(dr, dr) * dr
    F = F + torch.zeros_like(xv).index_add(1, v, visc).reshape(-1, 3) + st["load"].double().repeat(nc, 1)
    dt = float(np.float32(DT))
    u = pp[:, 3:] + F / 0.5 * dt
    return F, torch.cat([x + u * dt, u], 1)


def exact(case, seed):
    """no 64-bit counterpart for the flows between walls and with cells (the
    frozen walls and the order of the periodic images come from the framework),
    nor for runs long enough that a particle's cell can differ in 64 bits: the
    noise is drawn by position in the cell order, so one such particle gives all
    that follow it other noise"""
    kind, g = case["kind"], gen_of(seed, 1)
    if kind == "membranes":
        return membrane64(case, seed)
    if kind == "box" and case["rho"] * case["Lx"] * case["Ly"] * case["Lz"] * (case["steps"] - 1) <= 200_000:
        par = par64(*(case[k] for k in ("a", "g", "kBT", "dt", "spow")))
        return box64(box_size(case), fluid(box_size(case), case["rho"], case["kBT"], g), par, case["dt"], case["steps"])
    if kind == "forces":
        L = box_size(case)
        pp = fluid(L, case["rho"], case["kBT"], g)
        seeds = np.random.default_rng(seed).random(27).astype(np.float32).tolist()
        r, v, f = dpd64(L, pp[:, :3].double(), pp[:, 3:].double(),
                        par64(*(case[k] for k in ("a", "g", "kBT", "dt", "spow"))), seeds, 4)
        return torch.cat([r, v], 1), f
    if kind == "ensemble" and sum(b["rho"] * b["L"][0] * b["L"][1] * b["L"][2] for b in ensemble_boxes(case)) <= 60_000:
        out = []
        for k, b in enumerate(ensemble_boxes(case)):
            pp = fluid(b["L"], b["rho"], b["kBT"], gen_of(seed, 1, k))
            out.append(box64(b["L"], pp, par64(25.0, b["g"], b["kBT"], 1e-3, 0.25), 1e-3, case["steps"], 7919 * k)[0])
        return torch.cat(out)
    return None
