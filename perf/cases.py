"""The workloads the library's speed is measured on, each through its public entry points.

`listed()` names one case per way the library is used, from a 230-orbital deck
to the 762,112-orbital cell; `draw()` gives further cases of the same kinds
with sizes spread over the same ranges.  `prepare()` builds what a program
holds before the call (a handle with its geometry and Hamiltonian, networks,
input arrays), `run()` is one pass, `exact()` the same outputs in 64-bit torch
arithmetic on the prepared inputs, and `work()` the least bytes and operations
of a pass.

Kinds:
  deck      a whole small deck: geometry, pair search, every shift's job
            (assembly, local moments of the target orbitals, DoS)
  job       one k-point (or flake) job on a built geometry: assembly, block
            moments of random-phase vectors, DoS
  ldos      local moments of a few orbitals of a large flake (real H)
  trace     stochastic trace from caller-given real vectors (KPM_TRACE)
  bulk      moments of a block of random-phase vectors on a large matrix
  batch     many cells and k-points stacked in one recursion
  local     exact local moments of stacking configurations (the learned
            surrogate's fallback)
  cond      conductivity moments and their 2D transform
  dos       Jackson DoS of many moment rows
  train     Adam steps of one surrogate network
  ensemble  mean and spread of an ensemble of surrogate networks
"""
from __future__ import annotations

import math

import numpy as np
import torch

import leo2d_amd as L
from leo2d_amd import surrogate as S
from leo2d_amd import workloads as W

RESCALE = 10.5             # eV, above the Gershgorin bound of the GrapheneSimple bilayers
PER_AREA = 0.7531          # orbitals per A^2 of a bilayer disk
PER_ROW = 32.3             # stored entries per row of the pruned GrapheneSimple pattern
FULL_PER_ROW = 240.0       # slots per row of the full Graphene pattern away from a flake's edge
CACHE_BYTES = 32 << 20     # L2 of the eight XCDs: a recursion below this need not touch HBM per step


def listed():
    return [
        # the reference's own test deck: 230 orbitals, four shift jobs of local moments (smallest calls)
        {"name": "deck_230", "kind": "deck", "size": 10, "shifts": 2, "M": 200},
        # one Bloch k-point of the (7, 6) cell tiled 4 x 4, as a k-sampled deck or a small production job runs it
        {"name": "job_cell_8k", "kind": "job", "cell": 6, "tiles": 4, "R": 16, "M": 500, "bloch": True},
        # local DoS of the four centre orbitals of a 200 A disk, the reference's default observable
        {"name": "ldos_flake_95k", "kind": "ldos", "radius": 200.0, "R": 4, "M": 1024},
        # KPM_TRACE on a 100 A disk with the sample count such a deck takes by default (10^6 / n)
        {"name": "trace_flake_24k", "kind": "trace", "radius": 100.0, "R": 42, "M": 400},
        # the 1.05 degree cell tiled 4 x 4 at one k-point, 64 vectors in FP64
        {"name": "bulk_190k", "kind": "bulk", "cell": 31, "tiles": 4, "R": 64, "M": 512, "mixed": False},
        # the headline 762,112-orbital matrix with the FP32 recursion (largest)
        {"name": "bulk_762k_mixed", "kind": "bulk", "cell": 31, "tiles": 8, "R": 64, "M": 256, "mixed": True},
        # uneven commensurate cells at several k-points each in one stacked recursion
        {"name": "batch_cells", "kind": "batch", "cells": 8, "kpts": 4, "imin": 9, "imax": 31, "pick": 1, "R": 16,
         "M": 512, "mixed": False},
        # exact local moments where the surrogate's ensemble disagrees
        {"name": "local_sites", "kind": "local", "sites": 8, "theta_min": 1.0, "theta_max": 3.0, "pick": 3, "M": 512},
        # conductivity of the 200 A disk: four targets, 512 moments per direction
        {"name": "cond_flake_95k", "kind": "cond", "radius": 200.0, "R": 4, "M": 512},
        # DoS of a block of long moment rows (one per start vector or site)
        {"name": "dos_rows", "kind": "dos", "T": 32, "M": 4096},
        # training steps of one network on a batch of sites
        {"name": "surrogate_train", "kind": "train", "rows": 512, "hidden": 256, "out": 1024, "steps": 16},
        # spread of four networks over the sites of a flake
        {"name": "surrogate_sites", "kind": "ensemble", "rows": 32768, "hidden": 256, "out": 1024, "nets": 4,
         "mean": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _moments(rng, lo, hi):
    """A moment count: a multiple of 4."""
    return max(4, _log_int(rng, lo, hi) // 4 * 4)


def draw(rng):
    kind = rng.choice(["deck", "job", "job", "ldos", "ldos", "trace", "bulk", "bulk", "batch", "local", "cond", "dos",
                       "train", "ensemble"])
    if kind == "deck":
        return {"kind": kind, "size": rng.randint(6, 24), "shifts": rng.randint(1, 2), "M": _moments(rng, 64, 800)}
    if kind == "job":
        if rng.random() < 0.5:
            cell = rng.randint(4, 16)
            return {"kind": kind, "cell": cell, "tiles": rng.randint(1, max(1, 24 // cell)), "R": rng.randint(1, 40),
                    "M": _moments(rng, 100, 1000), "bloch": rng.random() < 0.75}
        return {"kind": kind, "radius": round(rng.uniform(25.0, 110.0), 2), "R": rng.randint(1, 40),
                "M": _moments(rng, 100, 800), "bloch": False}
    if kind == "ldos":
        return {"kind": kind, "radius": round(math.exp(rng.uniform(math.log(30.0), math.log(360.0))), 2),
                "R": rng.choice([1, 2, 2, 3, 4, 4, 6, 8]), "M": _moments(rng, 128, 1024)}
    if kind == "trace":
        return {"kind": kind, "radius": round(math.exp(rng.uniform(math.log(40.0), math.log(200.0))), 2),
                "R": rng.randint(4, 64), "M": _moments(rng, 100, 512)}
    if kind == "bulk":
        return {"kind": kind, "cell": rng.randint(24, 31), "tiles": rng.randint(2, 6), "R": rng.choice([16, 24, 32, 48, 64]),
                "M": _moments(rng, 64, 512), "mixed": rng.random() < 0.5}
    if kind == "batch":
        return {"kind": kind, "cells": rng.randint(2, 8), "kpts": rng.randint(1, 4), "imin": 5, "imax": 31,
                "pick": rng.randint(1, 10 ** 6), "R": rng.choice([4, 8, 16, 16, 32]), "M": _moments(rng, 100, 512),
                "mixed": rng.random() < 0.3}
    if kind == "local":
        return {"kind": kind, "sites": rng.randint(2, 10), "theta_min": 1.0, "theta_max": 3.0,
                "pick": rng.randint(1, 10 ** 6), "M": _moments(rng, 100, 512)}
    if kind == "cond":
        return {"kind": kind, "radius": round(math.exp(rng.uniform(math.log(30.0), math.log(200.0))), 2),
                "R": rng.randint(1, 4), "M": rng.randint(40, 512)}
    if kind == "dos":
        return {"kind": kind, "T": _log_int(rng, 1, 64), "M": _moments(rng, 64, 8192)}
    if kind == "train":
        return {"kind": kind, "rows": _log_int(rng, 64, 2048), "hidden": rng.choice([128, 200, 256, 384]),
                "out": rng.choice([256, 500, 1024, 2048]), "steps": rng.randint(2, 16)}
    return {"kind": "ensemble", "rows": _log_int(rng, 256, 32768), "hidden": rng.choice([128, 200, 256, 384]),
            "out": rng.choice([256, 500, 1024]), "nets": rng.randint(2, 4), "mean": rng.random() < 0.3}


# ---- inputs -------------------------------------------------------------------
def _small_deck(size, shifts, M, angle):
    sheet = "START_SHEET {s}\nMATERIAL = Graphene\nHEIGHT = {h}\nANGLE = {a!r}\nEND_SHEET {s}\n"
    return (f"JOB_NAME = small\nMAXSIZE = {size}\nMINSIZE = -{size}\nBOUNDARY_CONDITION = 0\nNUM_SHEETS = 2\n"
            + sheet.format(s=1, h=0, a=0.0) + sheet.format(s=2, h=3.4, a=angle)
            + f"SOLVER_TYPE = SQ\nNUM_TARGET_SHEETS = 2\nTARGET_SHEETS = 1 2\nNUM_SHIFT_SHEETS = 1\nSHIFT_SHEETS = 2\n"
              f"NSHIFTS = {shifts}\nENERGY_RESCALE = 13\nENERGY_SHIFT = 0.0\nPOLY_ORDER = {M}\n")


def _geometry(case):
    """The cell or flake a case runs on."""
    if "cell" in case:
        return L.Geometry(L.Deck(W.tblg_cell_deck(case["cell"] + 1, case["cell"], case["tiles"], M=case["M"])))
    return L.Geometry(L.Deck(W.tblg_flake_deck(1.05, case["radius"], M=case["M"], rescale=RESCALE)))


def _job(geom, rng, bloch):
    """The geometry's first job with a random shift of sheet 2, at a random k-point when bloch."""
    job = geom.jobs()[0]
    job.shift[1][0], job.shift[1][1] = float(rng.random()), float(rng.random())
    job.energy_rescale, job.energy_shift = RESCALE, 0.0
    if bloch:
        f = rng.random(2)
        k = f[0] * W.reciprocal(geom)[0] + f[1] * W.reciprocal(geom)[1]
        job.complex_matrix = 1
        job.k[0], job.k[1] = float(k[0]), float(k[1])
    else:
        job.complex_matrix = 0
    return job


def _ready(geom):
    dev = L.Device(0)
    dev.set_geometry(geom)
    dev.pairs_build()
    return dev


def _batch_cells(case):
    pick = np.random.default_rng(case["pick"])
    return [int(i) for i in pick.integers(case["imin"], case["imax"] + 1, size=case["cells"])]


def _batch_jobs(case, seed):
    """(geometry, job) of every stacked job."""
    rng = np.random.default_rng(seed)
    for i in _batch_cells(case):
        geom = L.Geometry(L.Deck(W.tblg_cell_deck(i + 1, i, M=case["M"])))
        yield geom, [_job(geom, rng, True) for _ in range(case["kpts"])]


def _site_cells(case):
    """The twists of a local case's sites (fixed by the case, not by the seed)."""
    pick = np.random.default_rng(case["pick"])
    th = np.exp(pick.uniform(math.log(case["theta_min"]), math.log(case["theta_max"]), case["sites"]))
    return [S.nearest_cell(t) for t in th]


def _network_inputs(rows, seed):
    rng = np.random.default_rng(seed)
    cfg = S.sample_configs(rows, rng, theta_range=(0.8, 3.0))
    return S.site_features(cfg, rng.integers(0, 4, rows)), rng


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if kind == "deck":
        return {"kind": kind, "dev": L.Device(0), "M": case["M"],
                "text": _small_deck(case["size"], case["shifts"], case["M"], float(rng.uniform(0.5, 30.0)))}
    if kind in ("job", "ldos", "trace", "cond"):
        geom = _geometry(case)
        dev = _ready(geom)
        job = _job(geom, rng, case.get("bloch", False))
        st = {"kind": kind, "dev": dev, "geom": geom, "job": job, "M": case["M"], "R": case["R"], "seed": seed}
        if kind == "ldos":
            dev.assemble(job, L.PATTERN_PRUNED)
            st["targets"] = rng.choice(geom.n, size=case["R"], replace=False).astype(np.int32)
        elif kind == "trace":
            dev.assemble(job, L.PATTERN_PRUNED)
            st["vectors"] = rng.standard_normal((case["R"], geom.n))
        elif kind == "cond":
            dev.assemble_velocity(job, L.PATTERN_PRUNED)
            st["targets"] = rng.choice(geom.n, size=case["R"], replace=False).astype(np.int32)
        return st
    if kind == "bulk":
        geom = _geometry(case)
        dev = _ready(geom)
        W.assemble_rescaled(dev, geom, rng.random(2))
        return {"kind": kind, "dev": dev, "geom": geom, "M": case["M"], "R": case["R"], "seed": seed,
                "precision": L.PREC_MIXED if case["mixed"] else L.PREC_FP64}
    if kind == "batch":
        dev = L.Device(0)
        for geom, jobs in _batch_jobs(case, seed):
            dev.set_geometry(geom)
            dev.pairs_build()
            for job in jobs:
                dev.assemble(job, L.PATTERN_PRUNED)
                dev.batch_append()
        return {"kind": kind, "dev": dev, "M": case["M"], "R": case["R"], "seed": seed,
                "precision": L.PREC_MIXED if case["mixed"] else L.PREC_FP64}
    if kind == "local":
        dev = L.Device(0)
        cells = _site_cells(case)
        cfg = np.column_stack([rng.random((len(cells), 2)), rng.normal(0.0, 0.003, (len(cells), 3)),
                               [S.cell_angle_deg(i) for i in cells]])
        return {"kind": kind, "exact": S.ExactLocalKPM(dev, case["M"]), "cfg": cfg,
                "blocks": rng.integers(0, 4, len(cells))}
    if kind == "dos":
        # moments of a smooth density: Jackson-damped decay with random phases
        n = np.arange(case["M"])
        mu = np.cos(rng.uniform(0, np.pi, (case["T"], 1)) * n) * np.exp(-n / rng.uniform(20, 500, (case["T"], 1)))
        return {"kind": kind, "dev": L.Device(0), "mu": mu}
    x, rng = _network_inputs(case["rows"], seed)
    if kind == "train":
        net = L.Mlp(0, S.N_IN, case["hidden"], 3, case["out"], seed=seed)
        return {"kind": kind, "net": net, "start": net.params(), "x": x, "steps": case["steps"],
                "t": rng.standard_normal((case["rows"], case["out"])).astype(np.float32)}
    nets = [L.Mlp(0, S.N_IN, case["hidden"], 3, case["out"], seed=seed * 16 + e) for e in range(case["nets"])]
    return {"kind": kind, "nets": nets, "x": x, "mean": case["mean"]}


# ---- one pass -------------------------------------------------------------------
def run(st):
    kind = st["kind"]
    if kind == "deck":
        dev = st["dev"]
        geom = L.Geometry(L.Deck(st["text"]))
        dev.set_geometry(geom)
        dev.pairs_build()
        mus, rhos = [], []
        for job in geom.jobs():
            dev.assemble(job, L.PATTERN_REFERENCE)
            mus.append(dev.kpm(st["M"], targets=list(job.targets[: job.num_targets])))
            rhos.append(dev.dos(mus[-1], job.energy_rescale, job.energy_shift)[1])
        return {"mu": np.array(mus), "rho": np.array(rhos)}
    if kind == "job":
        dev, job = st["dev"], st["job"]
        dev.assemble(job, L.PATTERN_PRUNED)
        mu = dev.kpm(st["M"], random_phase=(st["R"], st["seed"]), scheme=L.SCHEME_DOUBLING)
        E, rho = dev.dos(mu.mean(axis=0) / st["geom"].n, job.energy_rescale, job.energy_shift)
        return {"mu": mu, "E": E, "rho": rho}
    if kind == "ldos":
        return st["dev"].kpm(st["M"], targets=st["targets"])
    if kind == "trace":
        return st["dev"].kpm(st["M"], vectors=st["vectors"])
    if kind == "bulk":
        return st["dev"].kpm(st["M"], random_phase=(st["R"], st["seed"]), scheme=L.SCHEME_DOUBLING,
                             precision=st["precision"])
    if kind == "batch":
        return st["dev"].batch_kpm(st["M"], st["R"], seed=st["seed"], precision=st["precision"], tune=True)
    if kind == "local":
        return st["exact"].moments_at(st["cfg"], st["blocks"])
    if kind == "cond":
        C = st["dev"].cond_moments(st["M"], st["targets"])
        return {"C": C, "sigma": st["dev"].cond_transform(C)}
    if kind == "dos":
        E, rho = st["dev"].dos(st["mu"], RESCALE, 0.0)
        return {"E": E, "rho": rho}
    if kind == "train":
        st["net"].set_params(st["start"])
        losses = st["net"].train(st["x"], st["t"], epochs=st["steps"], batch=st["x"].shape[0])
        return {"losses": losses, "params": st["net"].params()}
    mean, spread = L.mlp_ensemble(st["nets"], st["x"], with_mean=st["mean"])
    return {"mean": mean, "spread": spread} if st["mean"] else {"spread": spread}


# ---- least work of a pass ---------------------------------------------------------
def _recursion(n, nnz, R, M, val, vec, flop):
    """M/2 steps of out = 2 H x - out on a block of R vectors."""
    matrix, block = nnz * (val + 4), n * R * vec
    steps = M // 2 if matrix + 2 * block > CACHE_BYTES else 1
    return {"bytes": float(steps * (matrix + 3 * block)), "flops": float(nnz) * R * flop * (M // 2)}


def _orbitals(case):
    if "cell" in case:
        return W.cell_orbitals(case["cell"]) * case["tiles"] ** 2
    return PER_AREA * math.pi * case["radius"] ** 2


def work(case):
    kind, M = case["kind"], case.get("M", 0)
    if kind == "deck":
        n = PER_AREA * math.pi * case["size"] ** 2
        per = min(0.65 * n, FULL_PER_ROW)
        w = _recursion(n, n * per, 2, M, 8, 8, 2)
        return {"bytes": case["shifts"] ** 2 * w["bytes"], "flops": case["shifts"] ** 2 * w["flops"]}
    if kind in ("job", "bulk"):
        n = _orbitals(case)
        cpx = kind == "bulk" or case["bloch"]
        half = 2 if case.get("mixed") else 1
        return _recursion(n, n * PER_ROW, case["R"], M, (16 if cpx else 8) // half, 16 // half, 8 if cpx else 4)
    if kind in ("ldos", "trace"):
        n = _orbitals(case)
        return _recursion(n, n * PER_ROW, case["R"], M, 8, 8, 2)
    if kind == "batch":
        n = case["kpts"] * sum(W.cell_orbitals(i) for i in _batch_cells(case))
        half = 2 if case["mixed"] else 1
        return _recursion(n, n * PER_ROW, case["R"], M, 16 // half, 16 // half, 8)
    if kind == "local":
        n = sum(W.cell_orbitals(i) for i in _site_cells(case))
        return _recursion(n, n * PER_ROW, 4, M, 8, 8, 2)
    if kind == "cond":
        n = _orbitals(case)
        R, nnz = case["R"], n * PER_ROW
        return {"bytes": 2.0 * n * R * M * 8 + nnz * 20, "flops": R * (3.0 * M * nnz * 2 + 2.0 * M * M * n + 4.0 * M ** 3)}
    if kind == "dos":
        T = case["T"]
        return {"bytes": 16.0 * T * M, "flops": 2.5 * T * M * math.log2(2 * M)}   # a fast cosine transform
    dims = [S.N_IN] + [case["hidden"]] * 3 + [case["out"]]
    params = sum(a * b + b for a, b in zip(dims, dims[1:]))
    fwd = 2.0 * sum(a * b for a, b in zip(dims, dims[1:])) * case["rows"]
    io = 4.0 * case["rows"] * S.N_IN
    if kind == "train":
        return {"bytes": io + 4.0 * case["rows"] * case["out"] + case["steps"] * params * 24.0,
                "flops": 3.0 * fwd * case["steps"]}
    return {"bytes": io + case["nets"] * params * 2.0 + 4.0 * case["rows"] * (1 + (case["out"] if case["mean"] else 0)),
            "flops": fwd * case["nets"]}


# ---- the same outputs in 64-bit arithmetic ------------------------------------------
def _torch_device():
    return torch.device("cuda:0" if torch.cuda.is_available() else "cpu")


def _padded(rp, ci, val):
    """CSR arrays as padded [longest][n] columns and values."""
    dv = _torch_device()
    rp, ci, val = (torch.from_numpy(a).to(dv) for a in (rp, ci, val))
    n = rp.numel() - 1
    lens = rp[1:] - rp[:-1]
    width = int(lens.max())
    rows = torch.repeat_interleave(torch.arange(n, device=dv), lens)
    at = (torch.arange(ci.numel(), device=dv) - rp[rows]) * n + rows
    cols = torch.zeros(width * n, dtype=torch.int64, device=dv)
    vals = torch.zeros(width * n, dtype=val.dtype, device=dv)
    cols[at] = ci.to(torch.int64)
    vals[at] = val
    return cols.reshape(width, n), vals.reshape(width, n)


def _apply(H, x):
    cols, vals = H
    y = torch.zeros_like(x)
    for c, v in zip(cols, vals):
        y += v[:, None] * x[c]
    return y


def _moments64(H, v0, M, segment=None, jobs=1):
    """<v|T_n(H)|v> of every column of v0 (per segment of rows), by products of T_j and T_{j+1}."""
    if v0.is_complex() and not H[1].is_complex():
        H = (H[0], H[1].to(v0.dtype))
    elif H[1].is_complex() and not v0.is_complex():
        v0 = v0.to(H[1].dtype)

    def dots(a, b):
        p = (a.conj() * b).real if a.is_complex() else a * b
        if segment is None:
            return p.sum(0, keepdim=True)
        return torch.zeros(jobs, p.shape[1], dtype=p.dtype, device=p.device).index_add_(0, segment, p)

    a, b = v0, _apply(H, v0)
    mu0, mu1 = dots(a, a), dots(b, a)
    mu = [mu0, mu1]
    for _ in range(1, M // 2):
        a, b = b, 2 * _apply(H, b) - a
        mu += [2 * dots(a, a) - mu0, 2 * dots(b, a) - mu1]
    return torch.stack(mu, dim=2).cpu().numpy()      # [jobs][R][M]


def _mix(z):
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


def _random_phases(seed, first, R, n):
    """The library's random-phase vectors first .. first + R - 1 on n orbitals (splitmix64 of seed, vector, orbital)."""
    with np.errstate(over="ignore"):
        h = _mix(np.uint64(seed) * np.uint64(0x9E3779B97F4A7C15) + np.uint64(0x632BE59BD9B4E019))
        hr = _mix(h ^ (np.arange(first, first + R, dtype=np.uint64) * np.uint64(0xD1B54A32D192ED03)))
        hi = _mix(hr[None, :] ^ (np.arange(n, dtype=np.uint64)[:, None] * np.uint64(0x8CB92BA72F3D8DD7)))
    phi = (hi >> np.uint64(11)).astype(np.float64) * (1.0 / 9007199254740992.0) * 6.283185307179586
    return torch.from_numpy(np.exp(1j * phi)).to(_torch_device())


def _unit(n, targets):
    v = torch.zeros(n, len(targets), dtype=torch.float64, device=_torch_device())
    v[torch.as_tensor(np.asarray(targets), dtype=torch.int64), torch.arange(len(targets))] = 1.0
    return v


def _cond64(H, D, targets, M):
    n = H[0].shape[1]
    e = _unit(n, targets)

    def chebyshev(x):
        out, a, b = [x], x, _apply(H, x)
        for _ in range(1, M):
            out.append(b)
            a, b = b, 2 * _apply(H, b) - a
        return torch.stack(out[:M])                  # [M][n][R]

    beta = chebyshev(e)
    alpha = chebyshev(-_apply(D, e))
    C = torch.stack([torch.stack([_apply(D, a[:, r:r + 1])[:, 0] for a in alpha]) @ beta[:, :, r].T
                     for r in range(len(targets))])
    i = torch.arange(M, dtype=torch.float64, device=C.device)
    g = ((M - i) * torch.cos(math.pi * i / M) + torch.sin(math.pi * i / M) / math.tan(math.pi / M)) / (math.sqrt(2.0) * M)
    phase = torch.remainder(torch.arange(M, device=C.device)[None, :] * (2 * torch.arange(M, device=C.device)[:, None] + 1),
                            4 * M).to(torch.float64)
    P = 2 * torch.cos(math.pi * phase / (2 * M))
    P[:, 0] = 1.0
    sigma = torch.stack([P @ (2 * g[:, None] * g[None, :] * c) @ P.T for c in C])
    return {"C": C.cpu().numpy(), "sigma": sigma.cpu().numpy()}


def _dos64(mu, a):
    T, M = mu.shape
    n = np.arange(M)
    g = ((M - n) * np.cos(np.pi * n / M) + np.sin(np.pi * n / M) / np.tan(np.pi / M)) / M
    w = torch.from_numpy(g * mu * np.where(n == 0, 1.0, 2.0)).to(_torch_device())
    cos = torch.cos(torch.arange(4 * M, device=w.device, dtype=torch.float64) * (math.pi / (2 * M)))
    k, i = torch.arange(M, device=w.device), torch.arange(M, device=w.device)
    out = torch.cat([w @ cos[torch.remainder(i[:, None] * (2 * kk[None, :] + 1), 4 * M)] for kk in k.split(512)], dim=1)
    E = a * np.cos((n + 0.5) * np.pi / M)
    return {"E": E, "rho": out.cpu().numpy() / (np.pi * np.sqrt(a * a - E * E))}


def _network64(p, dims):
    """Weights and biases of a flat parameter vector."""
    out, at = [], 0
    for a, b in zip(dims, dims[1:]):
        out += [p[at:at + a * b].reshape(b, a), p[at + a * b:at + a * b + b]]
        at += a * b + b
    return out


def _forward64(wb, x):
    for k in range(0, len(wb) - 2, 2):
        x = torch.nn.functional.gelu(x @ wb[k].T + wb[k + 1], approximate="tanh")
    return x @ wb[-2].T + wb[-1]


def _train64(st, lr=1e-3, b1=0.9, b2=0.999, eps=1e-8):
    dv = _torch_device()
    p = torch.from_numpy(st["start"]).to(dv).double()
    x, t = torch.from_numpy(st["x"]).to(dv).double(), torch.from_numpy(st["t"]).to(dv).double()
    m, v, losses = torch.zeros_like(p), torch.zeros_like(p), []
    for k in range(1, st["steps"] + 1):
        p.requires_grad_(True)
        loss = (_forward64(_network64(p, st["net"].dims), x) - t).square().mean()
        g, = torch.autograd.grad(loss, p)
        losses.append(float(loss))
        p = p.detach()
        m, v = b1 * m + (1 - b1) * g, b2 * v + (1 - b2) * g * g
        p = p - lr * (m / (1 - b1 ** k)) / ((v / (1 - b2 ** k)).sqrt() + eps)
    return {"losses": np.array(losses), "params": p.cpu().numpy()}


def _ensemble64(st):
    x = torch.from_numpy(st["x"]).to(_torch_device()).double()
    nets = [_network64(torch.from_numpy(m.params()).to(x.device).double(), m.dims) for m in st["nets"]]
    mean, spread = [], []
    for rows in x.split(4096):
        y = torch.stack([_forward64(wb, rows) for wb in nets])
        mean.append(y.mean(0))
        spread.append(y.var(0, unbiased=False).mean(1).sqrt())
    out = {"spread": torch.cat(spread).cpu().numpy()}
    if st["mean"]:
        out["mean"] = torch.cat(mean).cpu().numpy()
    return out


def exact(case, seed):
    """The outputs of run() from the prepared inputs (a handle's Hamiltonian among them) in 64 bits.

    deck, job and local cases assemble inside run(): their Hamiltonian is not an
    input, so they have no value computed without the library."""
    kind = case["kind"]
    if kind in ("deck", "job", "local"):
        return None
    if kind == "batch":
        R, rows, parts, starts, segment = case["R"], 0, [], [], []
        dev = L.Device(0)
        p = 0
        for geom, jobs in _batch_jobs(case, seed):
            dev.set_geometry(geom)
            dev.pairs_build()
            for job in jobs:
                dev.assemble(job, L.PATTERN_PRUNED)
                cols, vals = _padded(*dev.csr_copy())
                parts.append((cols + rows, vals))
                starts.append(_random_phases(seed, p * R, R, geom.n))
                segment.append(torch.full((geom.n,), p, dtype=torch.int64, device=cols.device))
                rows += geom.n
                p += 1
        width = max(c.shape[0] for c, _ in parts)
        pad = [(torch.nn.functional.pad(c, (0, 0, 0, width - c.shape[0])),
                torch.nn.functional.pad(v, (0, 0, 0, width - v.shape[0]))) for c, v in parts]
        H = torch.cat([c for c, _ in pad], dim=1), torch.cat([v for _, v in pad], dim=1)
        return _moments64(H, torch.cat(starts), case["M"], torch.cat(segment), p)
    st = prepare(case, seed)
    if kind == "dos":
        return _dos64(st["mu"], RESCALE)
    if kind == "train":
        return _train64(st)
    if kind == "ensemble":
        return _ensemble64(st)
    rp, ci, val = st["dev"].csr_copy()
    H = _padded(rp, ci, val)
    n = len(rp) - 1
    if kind == "cond":
        return _cond64(H, _padded(rp, ci, st["dev"].velocity_copy()), st["targets"], case["M"])
    if kind == "ldos":
        return _moments64(H, _unit(n, st["targets"]), case["M"])[0]
    if kind == "trace":
        return _moments64(H, torch.from_numpy(st["vectors"].T.copy()).to(_torch_device()), case["M"])[0]
    return _moments64(H, _random_phases(seed, 0, case["R"], n), case["M"])[0]
