"""The work that users of this framework have it do, as cases to be timed.

Every case goes through the Python entry points (`FMM`, `bem`) with its
inputs in HBM.  The mixed engine computes in FP32 and returns its sums in
FP64 containers; the programs these cases stand for keep their particles in
FP32 and take such results back to FP32.  Results of the FP64 engine and of
the direct sum stay FP64.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import old_fmm_bem_amd as F
from old_fmm_bem_amd import bem, workloads

DEV = "cuda"
# pairs of a direct sum in 64 bits that torch works through in a few seconds
EXACT_PAIRS = 1.0e11


def listed():
    return [
        # one-shot call on a handful of points (a unit test, the small
        # molecules of the BEM application): launches and latency only
        {"name": "cube_1k", "kind": "cube", "n": 1000, "p": 6, "lmax": 0, "precision": "mixed"},
        # the order and size of an everyday run; nothing about the tree given
        {"name": "cube_100k", "kind": "cube", "n": 100003, "p": 8, "lmax": 0, "precision": "mixed"},
        # the benchmark's headline step: 1M points, order 10, tree and matvec
        {"name": "cube_1m", "kind": "cube", "n": 1000000, "p": 10, "lmax": 5, "precision": "mixed"},
        # the largest step of the automatic depth's fitted range
        {"name": "cube_3m", "kind": "cube", "n": 3000000, "p": 10, "lmax": 0, "precision": "mixed"},
        # the FP64 engine, as a run that needs more than FP32 has it
        {"name": "cube_250k_fp64", "kind": "cube", "n": 250000, "p": 10, "lmax": 0, "precision": "fp64"},
        # the reference's own convention and order (its test driver's
        # softened kernel with the self pair), for users who compare with it
        {"name": "ref_60k", "kind": "ref", "n": 60000, "p": 9, "lmax": 0, "precision": "mixed"},
        # one GMRES iteration of a boundary-element solve: the tree is kept,
        # single and double layer on the Gauss points of a sphere
        {"name": "bem_sphere", "kind": "layers", "n": 245760, "p": 10, "lmax": 5, "precision": "mixed"},
        # many small surfaces in one tree, one iteration's matvec of the
        # batched solver (the captured evaluation)
        {"name": "bem_batch", "kind": "batch", "surfaces": 12, "nmin": 1000, "nmax": 20000, "p": 8},
        # oscillatory Helmholtz on the unit sphere, the benchmark's size
        {"name": "helmholtz_1m", "kind": "helmholtz", "n": 1000000, "p": 12, "lmax": 0, "k": 5.0},
        # screened (Yukawa) electrostatics with forces
        {"name": "yukawa_300k", "kind": "yukawa", "n": 300000, "p": 8, "lmax": 0, "lam": 2.0},
        # a training step through the potential: forward and all gradients,
        # clustered sources and separate targets
        {"name": "plummer_gradients", "kind": "gradients", "n": 120000, "m": 90001, "p": 8, "lmax": 0},
        # validation of a run against the direct sum on sampled targets
        {"name": "direct_2k", "kind": "direct", "n": 2000, "m": 300000},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["cube", "cube", "cube", "cube", "ref", "layers", "batch", "helmholtz", "yukawa", "gradients",
                       "direct"])
    if kind == "cube":
        if rng.random() < 0.35:
            return {"kind": kind, "n": _log(rng, 1000, 400000), "p": rng.choice([6, 8, 10, 12]), "lmax": 0,
                    "precision": "fp64"}
        return {"kind": kind, "n": _log(rng, 500, 2000000), "p": rng.choice([6, 7, 8, 9, 10, 11, 12]), "lmax": 0,
                "precision": "mixed"}
    if kind == "ref":
        return {"kind": kind, "n": _log(rng, 1000, 100000), "p": rng.choice([6, 8, 9, 10]), "lmax": 0,
                "precision": rng.choice(["mixed", "fp64"])}
    if kind == "layers":
        return {"kind": kind, "n": _log(rng, 5000, 400000), "p": rng.choice([8, 10]), "lmax": 0, "precision": "mixed"}
    if kind == "batch":
        return {"kind": kind, "surfaces": rng.randint(2, 12), "nmin": 500, "nmax": _log(rng, 2000, 20000), "p": 8}
    if kind == "helmholtz":
        return {"kind": kind, "n": _log(rng, 10000, 700000), "p": rng.choice([8, 10, 12]), "lmax": 0,
                "k": rng.choice([2.0, 4.0, 5.0])}
    if kind == "yukawa":
        return {"kind": kind, "n": _log(rng, 5000, 400000), "p": rng.choice([6, 8, 10]), "lmax": 0,
                "lam": rng.choice([1.0, 2.0, 5.0])}
    if kind == "gradients":
        return {"kind": kind, "n": _log(rng, 5000, 150000), "m": _log(rng, 5000, 150000), "p": rng.choice([6, 8, 10]),
                "lmax": 0}
    return {"kind": "direct", "n": _log(rng, 64, 4000), "m": _log(rng, 10000, 300000)}


def _cols(x):
    return tuple(torch.from_numpy(np.ascontiguousarray(x[:, k])).to(DEV) for k in range(3))


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def _shell(n, rng):
    """Quasi-uniform points on the unit sphere (a jittered Fibonacci lattice),
    as the Gauss points of a triangulated sphere are."""
    k = np.arange(n) + rng.uniform(0.2, 0.8, n)
    z = 1 - 2 * k / n
    r = np.sqrt(np.maximum(0.0, 1 - z * z))
    ph = math.pi * (1 + 5 ** 0.5) * (np.arange(n) + 0.5) + rng.uniform(0, 2 * math.pi)
    return np.stack([r * np.cos(ph), r * np.sin(ph), z], 1).astype(np.float32)


def _inputs(case, seed):
    """numpy inputs of a case, from the seed alone"""
    kind, rng = case["kind"], np.random.default_rng(seed)
    if kind in ("cube", "ref", "yukawa"):
        x, q = workloads.cube(case["n"], seed)
        return {"x": x, "q": q}
    if kind == "layers":
        x = _shell(case["n"], rng)
        c = rng.standard_normal((3, 3))
        sig = 1.0 + x.astype(np.float64) @ c[0] + (x.astype(np.float64) ** 2) @ c[1] + (x.astype(np.float64) ** 3) @ c[2]
        return {"x": x, "q": (4 * math.pi / case["n"] * sig).astype(np.float32)}
    if kind == "helmholtz":
        x, q = workloads.sphere(case["n"], seed)
        return {"x": x, "q": q}
    if kind == "gradients":
        xj, q = workloads.plummer(case["m"], seed)
        xi, _ = workloads.plummer(case["n"], seed + 7919)
        return {"xi": xi, "xj": xj, "q": q, "w": rng.standard_normal(case["n"]).astype(np.float32)}
    if kind == "direct":
        x, q = workloads.cube(case["m"], seed)
        return {"xi": x[rng.permutation(case["m"])[:case["n"]]], "xj": x, "q": q}
    raise ValueError(kind)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        # panel counts spread evenly over the logarithm of their range; the
        # shapes (semi-axes, bumps) are the seed's
        rng = np.random.default_rng(seed)
        ns, surfaces = case["surfaces"], []
        for k in range(ns):
            npan = int(case["nmin"] * (case["nmax"] / case["nmin"]) ** ((k + 0.5) / ns))
            bumps = [(u / np.linalg.norm(u), rng.uniform(0, 0.1), rng.uniform(0.15, 0.4))
                     for u in rng.standard_normal((20, 3))]
            surfaces.append(bem.ellipsoid_surface(npan, rng.uniform(0.5, 2.0, 3), bumps))
        op = bem.BatchedInducedCharge(surfaces, p=case["p"], precision="mixed")
        return {"kind": kind, "op": op, "x": torch.from_numpy(rng.uniform(0.5, 1.5, op.n)).to(DEV)}
    a = _inputs(case, seed)
    s = {"kind": kind, "q": _dev(a["q"])}
    if kind in ("cube", "ref"):
        # the root cube is known beforehand, the points are new at each step
        s["f"] = F.FMM(p=case["p"], lmax=case["lmax"], precision=case["precision"],
                       convention="ref" if kind == "ref" else "exact", box=(0, 0, 0, 1))
        s["x"] = _cols(a["x"])
        s["double"] = case["precision"] == "fp64"
    elif kind == "yukawa":
        s["f"] = F.FMM(p=case["p"], lmax=case["lmax"], precision="mixed", box=(0, 0, 0, 1), lam=case["lam"])
        s["x"] = _cols(a["x"])
    elif kind == "helmholtz":
        s["f"] = F.FMM(p=case["p"], lmax=case["lmax"], precision="mixed", box=(-1.0, -1.0, -1.0, 2.00001), k=case["k"])
        s["x"] = _cols(a["x"])
    elif kind == "layers":
        # the tree of the surface stays for the whole solve
        s["f"] = F.FMM(p=case["p"], lmax=case["lmax"], precision=case["precision"])
        x = _dev(a["x"])
        s["f"].set_points(x, ni_normals=x, nj_normals=x)
    elif kind == "gradients":
        s["f"] = F.FMM(p=case["p"], lmax=case["lmax"], precision="mixed")
        s["xi"], s["xj"], s["w"] = _dev(a["xi"]), _dev(a["xj"]), _dev(a["w"])
    else:
        s["f"] = F.FMM(p=10, precision="fp64")
        s["xi"], s["xj"] = _dev(a["xi"]), _dev(a["xj"])
    return s


def run(s):
    kind = s["kind"]
    if kind == "batch":
        return s["op"].matvec(s["x"]).float()
    f = s["f"]
    if kind in ("cube", "ref", "yukawa"):
        f.set_points(s["x"])
        v, g = f.evaluate(s["q"], neq=F.YUKAWA if kind == "yukawa" else F.G)
        if s.get("double"):
            return {"v": v, "g": g}
        return {"v": v.float(), "g": g.float()}
    if kind == "helmholtz":
        f.set_points(s["x"])
        return f.evaluate(s["q"], neq=F.HELMHOLTZ)[0].to(torch.complex64)
    if kind == "layers":
        single, _ = f.evaluate(s["q"], neq=F.G, gradient=False)
        double, _ = f.evaluate(s["q"], neq=F.GNJ)
        return {"single": single.float(), "double": double.float()}
    if kind == "gradients":
        f.set_points(s["xi"], s["xj"])
        v, _ = f.evaluate(s["q"], gradient=False)
        dq, dxi, dxj = f.gradients(s["q"], s["w"])
        return {"v": v.float(), "dq": dq.float(), "dxi": dxi.float(), "dxj": dxj.float()}
    v, g = f.direct(s["xi"], s["xj"], s["q"])
    return {"v": v, "g": g}


def work(case):
    """Bytes: coordinates, charges and normals read once, results written
    once.  Operations: direct sums count 20 per pair (30 Yukawa, 40
    Helmholtz); an FMM counts its near field at about 30 points per leaf
    (27 leaves, 9 of a surface) and, per leaf, its interaction list (189
    boxes, 27 of a surface) at the 6 p^3 of a rotation-based translation."""
    kind = case["kind"]
    if kind == "direct":
        n, m = case["n"], case["m"]
        return {"bytes": 12 * n + 16 * m + 32 * n, "flops": 20 * n * m}
    surface = kind in ("layers", "helmholtz", "batch")
    near, far = (9, 27) if surface else (27, 189)
    pair = {"yukawa": 30, "helmholtz": 40}.get(kind, 20)
    if kind == "batch":
        n = case["surfaces"] * (case["nmax"] - case["nmin"]) / math.log(case["nmax"] / case["nmin"])
        b, evals = 8 * n + 12 * n + 12 * n + 4 * n, 1
    elif kind == "gradients":
        n = 0.5 * (case["n"] + case["m"])
        b, evals = 16 * case["n"] + 16 * case["m"] + 16 * case["n"] + 16 * case["m"], 2
    elif kind == "layers":
        n = case["n"]
        b, evals = 28 * n + 8 * n, 2
    else:
        n = case["n"]
        out = 32 if case.get("precision") == "fp64" else 16
        b, evals = 16 * n + out * n, 1
        if kind == "helmholtz":
            b = 20 * n + 8 * n
    leaf = 30.0
    translate = 6 * case["p"] ** 3 * (4 if kind == "helmholtz" else 1)
    flops = evals * (pair * near * leaf * n + far * (n / leaf) * translate)
    return {"bytes": int(b), "flops": int(flops)}


def _direct64(xi, xj, q, kernel, grad, soft=0.0, lam=0.0, nj=None):
    """Direct sum in 64 bits over blocks of targets: potential, gradient.
    Without softening, coincident pairs are left out."""
    n, m = xi.shape[0], xj.shape[0]
    v = torch.zeros(n, dtype=q.dtype, device=xi.device)
    g = torch.zeros((n, 3), dtype=torch.float64, device=xi.device) if grad else None
    blk = max(1, min(n, int(6e7 // max(1, m))))
    c4 = 0.25 / math.pi
    for a in range(0, n, blk):
        t = xi[a:a + blk]
        d = [t[:, k:k + 1] - xj[None, :, k] for k in range(3)]
        r2 = d[0] * d[0]
        r2.addcmul_(d[1], d[1]).addcmul_(d[2], d[2])
        if soft:
            r2 += soft
        inv = torch.rsqrt(r2)
        if not soft:
            inv.masked_fill_(r2 == 0, 0.0)
        if kernel == "laplace":
            v[a:a + blk] = c4 * (inv @ q)
            if grad:
                inv3 = inv * inv * inv
                for k in range(3):
                    g[a:a + blk, k] = -c4 * ((d[k] * inv3) @ q)
        elif kernel == "double":
            dot = d[0] * nj[None, :, 0] + d[1] * nj[None, :, 1] + d[2] * nj[None, :, 2]
            v[a:a + blk] = c4 * ((dot * inv * inv * inv) @ q)
        elif kernel == "yukawa":
            c = 0.5 * math.pi / lam
            r = r2 * inv
            e = torch.exp(-lam * r) * inv
            v[a:a + blk] = c * (e @ q)
            if grad:
                rs = e * (1 + lam * r) * inv * inv
                for k in range(3):
                    g[a:a + blk, k] = -c * ((d[k] * rs) @ q)
        else:
            r = r2 * inv
            ck, sk = torch.cos(lam * r) * inv, torch.sin(lam * r) * inv
            v[a:a + blk] = c4 * torch.complex(ck @ q.real - sk @ q.imag, sk @ q.real + ck @ q.imag)
    return v, g


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        return None
    n = case["n"]
    if float(n) * case.get("m", n) > EXACT_PAIRS:
        return None
    a = {k: _dev(x) for k, x in _inputs(case, seed).items()}
    q = a["q"].to(torch.complex128 if kind == "helmholtz" else torch.float64)
    if kind in ("cube", "ref", "yukawa"):
        x = a["x"].double()
        v, g = _direct64(x, x, q, "yukawa" if kind == "yukawa" else "laplace", True,
                         soft=float(np.float32(1e-6)) if kind == "ref" else 0.0, lam=case.get("lam", 0.0))
        return {"v": v, "g": g}
    if kind == "helmholtz":
        x = a["x"].double()
        return _direct64(x, x, q, "helmholtz", False, lam=case["k"])[0]
    if kind == "layers":
        x = a["x"].double()
        return {"single": _direct64(x, x, q, "laplace", False)[0],
                "double": _direct64(x, x, q, "double", False, nj=x)[0]}
    xi, xj = a["xi"].double(), a["xj"].double()
    v, g = _direct64(xi, xj, q, "laplace", True)
    if kind == "direct":
        return {"v": v, "g": g}
    w = a["w"].double()
    dq, gj = _direct64(xj, xi, w, "laplace", True)
    return {"v": v, "dq": dq, "dxi": w[:, None] * g, "dxj": q[:, None] * gj}
