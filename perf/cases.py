"""Performance cases of the FMM velocity library: what a user has it compute.

Every case is one solve through the Python entry points (``FmmSolver`` and
``VelocityCalc``), with inputs resident on the GPU, except the host-array case,
which goes through ``VelocityCalc.get_velocity`` as a host time loop does.  A
case is a dict of plain values:

* ``call``   -- the entry point: ``velocity`` (2-D velocity on device tensors),
  ``host`` (``VelocityCalc.get_velocity`` on numpy arrays), ``potential``,
  ``type1`` (the type-1 FMM), ``ring`` (the 3-D treecode);
* ``field``  -- the particle field: ``plate`` (impulsively started flat plate),
  ``shed`` (the plate with shed vortices), ``street`` (von Karman street),
  ``vortices`` (uniform grid, the quiet part inactive), ``clusters`` (random
  blob over a uniform background), ``ring`` (vortex ring);
* ``n``      -- the nominal particle count: the fields are grids whose spacing
  gives about this many particles, so the actual counts are odd and ragged;
* ``jitter`` -- displacement off the grid in units of the spacing: 0 just after
  remeshing, more after some advection steps;
* ``idle``   -- share of inactive particles of a ``clusters`` field;
* the solver's own options (precision, order, p, max_par, icutoff, ...).
"""
from __future__ import annotations

import math

import numpy as np
import torch

from lsmps_vpm_v2_amd import FmmSolver, workloads
from lsmps_vpm_v2_amd.solver import Particle, VelocityCalc

PLATE_N, PLATE_H = 779_280, 0.0025   # the flat plate's default size and row spacing
SHED_MIN = 1_000_000                 # the shed field is the default plate plus its vortices
STREET_MIN = 200_000                 # the street's body layer alone holds about 90,000
EXACT_MAX_2D, EXACT_MAX_REG, EXACT_MAX_3D = 800_000, 250_000, 150_000


def listed():
    return [
        # the smallest solves: a coarse start or a test run, where launches and
        # latency count (reference options: p 10, leaf rule 75/50)
        dict(name="fp64_clusters_2k", call="velocity", field="clusters", n=2_000, idle=0.1,
             jitter=0.0, precision="fp64", order="fixed", p=10, max_par=75, max_src=50,
             icutoff=0),
        # a host time loop through the drop-in class: the size of a
        # multiresolution field after adaptation, particles on and off
        dict(name="host_vortices_54k", call="host", field="vortices", n=54_400, jitter=0.0,
             p=10),
        # the parity path at the flat-plate size, reference options
        dict(name="fp64_plate_780k", call="velocity", field="plate", n=PLATE_N, jitter=0.0,
             precision="fp64", order="fixed", p=10, max_par=75, max_src=50, icutoff=0),
        # FP64 with the Gaussian near field (regularized blobs), ragged leaves
        dict(name="fp64_gauss_clusters_100k", call="velocity", field="clusters", n=100_003,
             idle=0.0, jitter=0.0, precision="fp64", order="fixed", p=10, max_par=75,
             max_src=50, icutoff=2),
        # the learned FP32/MFMA path: a small random field
        dict(name="learned_clusters_20k", call="velocity", field="clusters", n=20_011, idle=0.0,
             jitter=0.0, precision="mixed", order="learned", p=12, max_par=48, max_src=48,
             icutoff=0),
        # the benchmark workload: the remeshed flat plate, learned orders
        dict(name="learned_plate_780k", call="velocity", field="plate", n=PLATE_N, jitter=0.0,
             precision="mixed", order="learned", p=12, max_par=48, max_src=48, icutoff=0),
        # the same path between two remeshings, with shed vortices (2M particles)
        dict(name="learned_shed_2m", call="velocity", field="shed", n=2_000_000, jitter=0.3,
             precision="mixed", order="learned", p=12, max_par=48, max_src=48, icutoff=0),
        # the largest field: a von Karman street on a full background grid,
        # fixed order
        dict(name="mixed_street_8m", call="velocity", field="street", n=8_000_000, jitter=0.2,
             precision="mixed", order="fixed", p=8, max_par=96, max_src=96, icutoff=0),
        # the potential that the pressure solver asks for
        dict(name="potential_vortices_100k", call="potential", field="vortices", n=100_000,
             jitter=0.0, p=10),
        # the type-1 FMM (Gaussian blobs, the reference's L2L)
        dict(name="type1_plate_200k", call="type1", field="plate", n=200_000, jitter=0.3, lmax=9,
             ndp=10, n_s=50, icutoff=2),
        # the 3-D treecode: a moderate ring and the full-size one
        dict(name="ring_60k", call="ring", field="ring", n=60_000, jitter=0.25, type=2),
        dict(name="ring_780k", call="ring", field="ring", n=780_000, jitter=0.0, type=1),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))))) | 1


def draw(rng):
    kind = rng.choice(["fp64", "fp64", "learned", "mixed", "host", "potential", "type1", "ring"])
    jitter = rng.choice([0.0, round(rng.uniform(0.05, 0.5), 3)])
    if kind == "ring":
        return dict(call="ring", field="ring", n=_log_uniform(rng, 3_000, 700_000),
                    jitter=jitter, type=rng.choice([1, 2]))
    if kind == "type1":
        n = _log_uniform(rng, 5_000, 700_000)
        return dict(call="type1", field=rng.choice(["plate", "clusters"]), n=n, jitter=jitter,
                    idle=0.0, lmax=7 if n < 50_000 else rng.choice([8, 9, 10]),
                    ndp=rng.choice([8, 10, 12]), n_s=50, icutoff=rng.choice([1, 2, 2, 3]))
    if kind in ("host", "potential"):
        return dict(call=kind, field=rng.choice(["plate", "clusters", "vortices"]),
                    n=_log_uniform(rng, 2_000, 700_000), jitter=jitter,
                    idle=rng.choice([0.0, 0.1, 0.3]), p=rng.choice([8, 10, 12]))
    c = dict(call="velocity", jitter=jitter, idle=rng.choice([0.0, 0.1, 0.3]))
    if kind == "fp64":
        c.update(n=_log_uniform(rng, 1_000, 1_500_000), precision="fp64", order="fixed",
                 p=rng.choice([8, 10, 10, 12]), max_par=75, max_src=50,
                 icutoff=rng.choice([0, 0, 0, 1, 2, 3]))
    elif kind == "learned":
        c.update(n=_log_uniform(rng, 5_000, 2_500_000), precision="mixed", order="learned", p=12,
                 max_par=48, max_src=48, icutoff=0, idle=0.0)
    else:
        thr = rng.choice([32, 48, 64, 96])
        c.update(n=_log_uniform(rng, 2_000, 6_000_000), precision="mixed", order="fixed",
                 p=rng.choice([7, 8, 9, 10, 12]), max_par=thr, max_src=thr,
                 icutoff=rng.choice([0, 0, 0, 2]))
    fields = ["clusters"]
    if c["n"] <= 2_000_000:
        fields += ["plate", "vortices"]
    if c["n"] >= 2 * SHED_MIN and c["n"] <= 3_000_000:
        fields.append("shed")
    if c["n"] >= STREET_MIN:
        fields.append("street")
    c["field"] = rng.choice(fields)
    return c


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------
def _street(n, seed):
    """The von Karman street of ``workloads.von_karman`` (two staggered rows of
    Lamb-Oseen vortices behind a cylinder with a fine body layer), formed on
    the GPU; the seed moves the vortices by up to a third of a core."""
    dev, rng = "cuda", np.random.Generator(np.random.PCG64(seed))
    half, radius, layer, h_body, core, gamma, n_vort = 20.0, 0.5, 0.1, 0.002, 0.3, 1.5, 40
    f64 = dict(dtype=torch.float64, device=dev)
    bx, by = [], []
    for k in range(int(round(layer / h_body))):
        r = radius + (k + 0.5) * h_body
        m = int(round(2 * math.pi * r / h_body))
        th = (torch.arange(m, **f64) + 0.5) * (2 * math.pi / m) + rng.uniform(0, 2 * math.pi / m)
        bx.append(r * torch.cos(th))
        by.append(r * torch.sin(th))
    bx, by = torch.cat(bx), torch.cat(by)
    wb = torch.sign(by) * 10.0 * torch.exp(-(torch.hypot(bx, by) - radius) / 0.02)
    m = int(round(math.sqrt((n - len(bx)) / (1 - math.pi * (radius + layer) ** 2 / (2 * half) ** 2))))
    h = 2 * half / m
    c = -half + (torch.arange(m, **f64) + 0.5) * h
    gx, gy = c.repeat(m), c.repeat_interleave(m)
    keep = gx * gx + gy * gy >= (radius + layer) ** 2
    gx, gy = gx[keep], gy[keep]
    wg = torch.zeros_like(gx)
    for k in range(n_vort):
        cx = 1.5 + (k // 2) * half / (n_vort / 2) * 0.92 + (0.45 if k % 2 else 0.0)
        cy = 0.6 if k % 2 == 0 else -0.6
        cx, cy = cx + rng.uniform(-0.1, 0.1), cy + rng.uniform(-0.1, 0.1)
        a = (-gamma if k % 2 == 0 else gamma) / (math.pi * core * core)
        wg += a * torch.exp(-((gx - cx) ** 2 + (gy - cy) ** 2) / (core * core))
    return dict(x=torch.cat([bx, gx]), y=torch.cat([by, gy]),
                s=torch.cat([torch.full_like(bx, h_body), torch.full_like(gx, h)]),
                omega=torch.cat([wb, wg]))


def _planar(case, seed):
    """x, y, s, omega (float64) and active (uint8) on the GPU.  Inactive
    particles are the ones without vorticity, as a solver marks them."""
    kind, n = case["field"], case["n"]
    if kind == "street":
        f = _street(n, seed)
    else:
        if kind == "plate":
            f = workloads.boundary_layer(seed=seed, h0=PLATE_H * math.sqrt(PLATE_N / n))
        elif kind == "shed":
            f = workloads.shed_vortices(seed=seed, n_total=n)
        elif kind == "vortices":
            f = workloads.uniform_vortices(seed=seed, h=20.0 / math.sqrt(n))
        else:
            f = workloads.random_clusters(n, seed=seed, active_frac=1.0 - case["idle"])
        f = {k: torch.from_numpy(f[k]).cuda() for k in ("x", "y", "s", "omega", "active")}
    if kind == "vortices":
        f["active"] = (f["omega"].abs() > 1e-2).to(torch.uint8)
    elif kind != "clusters":
        f["active"] = torch.ones_like(f["x"], dtype=torch.uint8)
    f["omega"] = f["omega"] * f["active"]
    if case["jitter"]:
        g = torch.Generator(device="cuda").manual_seed(seed)
        for k in ("x", "y"):
            r = torch.rand(f[k].shape, generator=g, dtype=torch.float64, device="cuda")
            f[k] = f[k] + case["jitter"] * f["s"] * (r - 0.5)
    return f


def _ring(case, seed):
    f = workloads.vortex_ring(case["n"], jitter=case["jitter"], seed=seed)
    g = torch.Generator(device="cuda").manual_seed(seed)
    f = {k: torch.from_numpy(f[k]).cuda() for k in
         ("x", "y", "z", "s", "wx", "wy", "wz", "active")}
    # a few per cent of scatter in the vorticity, so that every field differs
    scale = 1 + 0.05 * (torch.rand(f["x"].shape, generator=g, dtype=torch.float64,
                                   device="cuda") - 0.5)
    for k in ("wx", "wy", "wz"):
        f[k] = f[k] * scale
    return f


def prepare(case, seed):
    call = case["call"]
    if call == "ring":
        f = _ring(case, seed)
        out = [torch.empty_like(f["x"]) for _ in range(3)]
        return dict(case=case, solver=FmmSolver(), f=f, out=out)
    f = _planar(case, seed)
    if call == "host":
        h = {k: v.cpu().numpy() for k, v in f.items()}
        return dict(case=case, tool=VelocityCalc(p=case["p"]),
                    particle=Particle(h["x"], h["y"], h["s"], h["omega"], h["active"]))
    st = dict(case=case, f=f, out=[torch.empty_like(f["x"]) for _ in range(2)])
    if call == "velocity":
        mixed = case["precision"] == "mixed"
        st["solver"] = FmmSolver(p=case["p"], max_par=case["max_par"], max_src=case["max_src"],
                                 precision=case["precision"], order=case["order"],
                                 binom_mode=0 if mixed else 1, list4_mode=2 if mixed else 1,
                                 icutoff=case["icutoff"])
    elif call == "potential":
        f["q"] = -f["omega"] * f["s"] ** 2 / (2 * math.pi)
        st["solver"] = FmmSolver(p=case["p"])
    else:
        f["gz"] = f["omega"] * f["s"] ** 2
        st["solver"] = FmmSolver()
    return st


def run(state):
    case = state["case"]
    call = case["call"]
    if call == "host":
        p = state["particle"]
        state["tool"].get_velocity(p)
        return p.u, p.v
    f, s, out = state["f"], state["solver"], state["out"]
    if call == "ring":
        return s.velocity3d_device(f["x"], f["y"], f["z"], f["s"], f["wx"], f["wy"], f["wz"],
                                   f["active"], *out, type=case["type"])
    if call == "potential":
        return s.potential_device(f["x"], f["y"], f["q"], f["active"], out[0])
    if call == "type1":
        return s.velocity_type1_device(f["x"], f["y"], f["s"], f["gz"], *out, n_s=case["n_s"],
                                       lmax=case["lmax"], ndp=case["ndp"],
                                       icutoff=case["icutoff"])
    return s.velocity_device(f["x"], f["y"], f["s"], f["omega"], f["active"], *out)


# --------------------------------------------------------------------------
# what a pass cannot do without, and how far results may differ
# --------------------------------------------------------------------------
def work(case):
    """Bytes: every input read once, every output written once.  Flops: of the
    method, per particle -- 11 per pair with the nine neighbour leaves of mean
    occupancy m, and 27 translations of 8 (p + 1)^2 per cell (4/3 cells per
    leaf); in 3-D 26 per direct pair and 198 per far-cell term, 700 pairs and
    110 terms per octree level."""
    n, call = case["n"], case["call"]
    if call == "ring":
        return {"bytes": n * (7 * 8 + 1 + 3 * 8),
                "flops": n * (26 * 700 + 198 * 110 * math.log(max(n / 30, 8), 8))}
    m = 0.4 * {"velocity": case.get("max_src", 50), "type1": case.get("n_s", 50)}.get(call, 50)
    p = case["ndp"] if call == "type1" else case["p"]
    flops = n * (11 * 9 * m + 27 * 8 * (p + 1) ** 2 * (4 / 3) / m)
    arrays = {"potential": 4, "type1": 6}.get(call, 6)
    return {"bytes": n * (8 * arrays + (0 if call == "type1" else 1)), "flops": flops}


def tolerance(case):
    """Measured by permuting the particles, which reorders the sums inside
    every leaf: the FP64 paths differ by up to 9e-15 (largest single value
    4e-14), and the matrix-core M2L from the plain one by up to 9e-15 of the
    velocity, ten times that of the small component; the FP32 paths by up to
    3e-7 (largest single value 4.4e-6), with the same roundings of positions
    and expansions."""
    if case.get("precision") == "mixed":
        return {"rel": 1.5e-6, "max": 2e-5}
    return {"rel": 4e-13, "max": 4e-12}


def _direct2d(f, q, sizes=None, icutoff=0):
    """sum_j q_j / (z_i - z_j) over j != i (conjugate field), optionally with
    the regularization factor of the near-field kernels on every pair."""
    z = torch.complex(f["x"], f["y"])
    n = len(z)
    w = torch.complex(q, torch.zeros_like(q))
    out = torch.empty_like(z)
    step = max(1, (1 << 27) // n)
    for i in range(0, n, step):
        d = z[i:i + step, None] - z[None, :]
        rows = torch.arange(len(d), device=d.device)
        d[rows, rows + i] = 1.0
        if icutoff:
            r2 = d.real ** 2 + d.imag ** 2
            rho2 = r2 / (0.25 * (sizes[i:i + step, None] ** 2 + sizes[None, :] ** 2))
            if icutoff == 1:
                k = rho2 * (rho2 + 2) / (rho2 + 1) ** 2
            elif icutoff == 2:
                k = -torch.expm1(-0.5 * rho2)
            else:
                k = -torch.expm1(-0.5 * rho2) - 0.5 * rho2 * torch.exp(-0.5 * rho2)
            inv = k / d
        else:
            inv = d.reciprocal_()
        inv[rows, rows + i] = 0.0
        out[i:i + step] = inv @ w
    return out


def exact(case, seed):
    """The direct sum in 64 bits (None where it would take too long)."""
    call, n = case["call"], case["n"]
    if call == "ring":
        if n > EXACT_MAX_3D:
            return None
        f = _ring(case, seed)
        P = torch.stack([f["x"], f["y"], f["z"]], 1)
        A = torch.stack([f["wx"], f["wy"], f["wz"]], 1) * (f["s"] ** 3 / (4 * math.pi))[:, None]
        out = torch.empty_like(P)
        step = max(1, (1 << 25) // len(P))
        for i in range(0, len(P), step):
            d = P[i:i + step, None, :] - P[None, :, :]
            r2 = (d * d).sum(2)
            rows = torch.arange(len(d), device=d.device)
            r2[rows, rows + i] = math.inf
            # alpha x r / |r|^3, with r from the source to the target
            out[i:i + step] = (torch.linalg.cross(A[None].expand_as(d), d)
                               * (r2 ** -1.5)[:, :, None]).sum(1)
        return out[:, 0] + 1.0, out[:, 1].clone(), out[:, 2].clone()
    icut = case.get("icutoff", 0)
    if n > (EXACT_MAX_REG if icut or call == "potential" else EXACT_MAX_2D):
        return None
    f = _planar(case, seed)
    q = -f["omega"] * f["s"] ** 2 / (2 * math.pi)
    if call == "potential":
        m = len(q)
        out = torch.empty_like(q)
        step = max(1, (1 << 27) // m)
        for i in range(0, m, step):
            dx = f["x"][i:i + step, None] - f["x"][None, :]
            dy = f["y"][i:i + step, None] - f["y"][None, :]
            r2 = dx * dx + dy * dy
            rows = torch.arange(len(r2), device=r2.device)
            r2[rows, rows + i] = 1.0
            out[i:i + step] = 0.5 * (torch.log(r2) @ q)
        return out
    e = _direct2d(f, q, f["s"], icut)   # ex - i ey
    u, v = -e.imag + 1.0, -e.real.clone()
    if call == "host":
        return u.cpu().numpy(), v.cpu().numpy()
    return u, v
