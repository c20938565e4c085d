"""The work that users of this framework have it do, for timing and for comparing results.

Every case is one call a program makes: a system of bodies (or panels) with new positions or strengths goes in, the
field at its targets comes out. Sizes and settings are those of the repository's benchmark (bench.py: the 1M vortex
ring, the Plummer sweep, the batch of uneven systems, the serving stream's evaluations and panel solves) and of its
tests; the smallest calls are the sizes of a single small request.

A time-stepping program keeps one evaluation handle per system and calls set_systems + fmm + targets at every step;
that is what run() does for the device-resident cases. Systems handed over as objects (F.fmm, F.direct,
F.FastGaussSeidel) go through host arrays, as their interface has it.
"""
import math

import numpy as np
import torch

import fastmultipole_amd as F
from fastmultipole_amd import _lib, workloads as W

DEVICE = "cuda" if torch.cuda.is_available() else "cpu"
CORE = 0.1          # Gaussian core of the vortex ring's cross-section (bench.py)
EXACT_PAIRS = 1.0e11  # body pairs above which the direct sum in plain torch takes too long


# ------------------------------------------------------------------------------------------------------- cases
def listed():
    return [
        # one small request: 1,000 vortex particles handed over as a system object, fixed order, velocity + gradient
        dict(name="system_vortex_1k", kind="system", n=1000, p=8, leaf=20, mac=0.5),
        # the plain evaluation: 10,000 point sources in the unit cube, potential + gradient
        dict(name="cube_10k_p8", kind="fmm", dist="cube", n=10000, p=8, leaf=50, mac=0.5, tol=0.0, precision="fp64"),
        # a request of the serving stream's median size: vortex ring with a relative error tolerance
        dict(name="ring_45k_tol", kind="fmm", dist="ring", n=44721, p=20, leaf=64, mac=0.55, tol=1e-9, precision="fp64"),
        # a large system of the uneven batch, mixed precision, with the tolerance
        dict(name="ring_150k_tol_mixed", kind="fmm", dist="ring", n=150001, p=20, leaf=64, mac=0.55, tol=1e-9,
             precision="mixed"),
        # the headline: 1M-particle vortex ring, velocity + velocity gradient, order picked per interaction
        dict(name="ring_1m_tol", kind="fmm", dist="ring", n=1000000, p=20, leaf=64, mac=0.55, tol=1e-9, precision="fp64"),
        # the Plummer sweep's size at its middle order: strongly clustered sources, potential + gradient
        dict(name="plummer_4m_p8", kind="fmm", dist="plummer", n=4194304, p=8, leaf=50, mac=0.5, tol=0.0, precision="fp64"),
        # the sweep's highest order on a smaller sphere, mixed precision
        dict(name="plummer_300k_p16_mixed", kind="fmm", dist="plummer", n=300007, p=16, leaf=50, mac=0.5, tol=0.0,
             precision="mixed"),
        # uneven independent systems evaluated as one batch (cube sources, mixed precision, the tuned leaf size)
        dict(name="batch_48_cubes_mixed", kind="batch", systems=48, n_min=1000, n_max=100000, p=8, leaf=48, mac=0.5,
             precision="mixed"),
        # velocities at probe points away from the particles: regularised vortices as sources, separate targets
        dict(name="probes_100k_gaussian", kind="probes", n=100000, probes=131071, p=10, leaf=50, mac=0.5),
        # potential + velocity of a body's surface panels (quadrilaterals tiling a sphere)
        dict(name="panels_54k_quads", kind="panels", m=95, shape="source_quads", p=8, leaf=30, mac=0.5),
        # a serving stream's panel solve: set up and solve for the strengths that cancel a normal velocity
        dict(name="solve_20k_quads", kind="solve", m=58, p=6, leaf=30, mac=0.5, tol=1e-8),
        # the direct sum, every body on every body: the accuracy reference, and the evaluation of systems without a tree
        dict(name="direct_65k_vortex", kind="direct", n=65537),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["system", "cube", "ring", "ring_mixed", "plummer", "batch", "probes", "panels", "solve", "direct"])
    if kind == "system":
        return dict(kind="system", n=_log(rng, 300, 5000), p=rng.choice([4, 6, 8, 10]), leaf=rng.randint(10, 50),
                    mac=rng.choice([0.4, 0.5]))
    if kind == "cube":
        precision = rng.choice(["fp64", "mixed"])
        return dict(kind="fmm", dist=rng.choice(["cube", "vortices"]), n=_log(rng, 2000, 200000), p=rng.randint(4, 12),
                    leaf=rng.randint(20, 90), mac=rng.choice([0.4, 0.5, 0.6]), tol=0.0, precision=precision)
    if kind == "ring":
        return dict(kind="fmm", dist="ring", n=_log(rng, 5000, 800000), p=20, leaf=rng.randint(40, 90),
                    mac=rng.choice([0.5, 0.55]), tol=rng.choice([1e-6, 1e-9]), precision="fp64")
    if kind == "ring_mixed":
        return dict(kind="fmm", dist="ring", n=_log(rng, 5000, 200000), p=20, leaf=rng.randint(40, 90),
                    mac=rng.choice([0.5, 0.55]), tol=rng.choice([1e-6, 1e-9]), precision="mixed")
    if kind == "plummer":
        p = rng.choice([4, 8, 16])
        return dict(kind="fmm", dist="plummer", n=_log(rng, 50000, 600000 if p == 16 else 3000000), p=p,
                    leaf=rng.randint(40, 80), mac=0.5, tol=0.0, precision="fp64")
    if kind == "batch":
        return dict(kind="batch", systems=rng.randint(8, 64), n_min=1000, n_max=_log(rng, 10000, 90000), p=8,
                    leaf=rng.randint(32, 64), mac=0.5, precision=rng.choice(["fp64", "mixed"]))
    if kind == "probes":
        return dict(kind="probes", n=_log(rng, 5000, 150000), probes=_log(rng, 5000, 200000), p=rng.randint(6, 12),
                    leaf=rng.randint(20, 80), mac=rng.choice([0.4, 0.5]))
    if kind == "panels":
        return dict(kind="panels", m=_log(rng, 20, 100),
                    shape=rng.choice(["source_quads", "source_triangles", "dipole_quads", "dipole_triangles"]),
                    p=rng.choice([6, 8]), leaf=rng.randint(20, 50), mac=0.5)
    if kind == "solve":
        return dict(kind="solve", m=_log(rng, 16, 70), p=rng.choice([4, 6]), leaf=rng.randint(20, 40), mac=0.5, tol=1e-8)
    return dict(kind="direct", n=_log(rng, 1000, 100000))


# ------------------------------------------------------------------------------------------------------ inputs
def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=DEVICE, dtype=torch.float64)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEVICE, dtype=torch.float64)


def _ring(g, n, core=0.0):
    """workloads.vortex_ring's distribution, made on the device: (n, 7) rows [x, y, z, core, Gamma]."""
    phi = _rand(g, n) * (2.0 * math.pi)
    c, s = torch.cos(phi), torch.sin(phi)
    rr = 1.0 + CORE * _randn(g, n)
    t = torch.stack([-s, c, torch.zeros_like(s)], 1) + 1e-3 * _randn(g, n, 3)
    return torch.cat([(rr * c)[:, None], (rr * s)[:, None], (CORE * _randn(g, n))[:, None],
                      torch.full((n, 1), core, device=DEVICE, dtype=torch.float64), t * (2.0 * math.pi / n)], 1).contiguous()


def _cube(g, n):
    b = torch.zeros(n, 5, device=DEVICE, dtype=torch.float64)
    b[:, :3] = _rand(g, n, 3)
    b[:, 4] = _rand(g, n)
    return b


def _vortices(g, n):
    b = torch.zeros(n, 7, device=DEVICE, dtype=torch.float64)
    b[:, :3] = _rand(g, n, 3)
    b[:, 4:7] = (2.0 * _rand(g, n, 3) - 1.5) * 2.0 / n
    return b


def _plummer(g, n, rmax=20.0):
    """workloads.plummer_sources' distribution (scale 1, truncated at rmax), by the inverse of its mass profile."""
    u = _rand(g, n) * (1.0 + rmax ** -2) ** -1.5
    r = 1.0 / torch.sqrt(torch.clamp(u, min=1e-12) ** (-2.0 / 3.0) - 1.0)
    v = _randn(g, n, 3)
    b = torch.zeros(n, 5, device=DEVICE, dtype=torch.float64)
    b[:, :3] = v * (r / v.norm(dim=1))[:, None]
    b[:, 4] = _randn(g, n)
    return b


def _core(n):
    """1.5 times the mean spacing of n particles in the ring's core."""
    return 1.5 * (2.0 * math.pi * 2.0 * math.pi * CORE ** 2 / n) ** (1.0 / 3.0)


def _kernel(dist):
    return _lib.POINT_SOURCE if dist in ("cube", "plummer") else _lib.POINT_VORTEX


def _bodies(case, seed):
    return {"cube": _cube, "vortices": _vortices, "ring": _ring, "plummer": _plummer}[case["dist"]](_generator(seed), case["n"])


def _batch_counts(case):
    """The benchmark's uneven sizes: log-uniform, drawn once."""
    u = np.random.default_rng(4).uniform(math.log(case["n_min"]), math.log(case["n_max"]), case["systems"])
    return np.floor(np.exp(u)).astype(np.int64)


def _probe_points(g, n):
    """Points of the box around the ring, where a wake is surveyed."""
    return ((_rand(g, n, 3) - 0.5) * torch.tensor([3.0, 3.0, 1.0], device=DEVICE, dtype=torch.float64)).contiguous()


def _panel_vertices(case, seed):
    """(vertices (n, nv, 3), strengths) of the panels tiling a unit sphere."""
    rows, _ = W.sphere_panels(case["m"], quads="quads" in case.get("shape", "source_quads"), seed=seed)
    return rows[:, 5:].reshape(len(rows), -1, 3), rows[:, 4]


def _panel_kernel(shape):
    return {"source_quads": _lib.PANEL_SOURCE_QUAD, "source_triangles": _lib.PANEL_SOURCE_TRI,
            "dipole_quads": _lib.PANEL_DIPOLE_QUAD, "dipole_triangles": _lib.PANEL_DIPOLE_TRI}[shape]


def _panel_buffer(case, seed):
    v, q = _panel_vertices(case, seed)
    return torch.from_numpy(W.panel_rows(v, q)).to(DEVICE).contiguous()


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("system", "direct"):
        b = _ring(_generator(seed), case["n"]).cpu().numpy()
        s = dict(kind=kind, case=case, system=F.VortexParticles(b[:, :3], b[:, 4:7]))
        if kind == "system":
            s["ev"] = F.Evaluation()
        return s
    if kind == "solve":
        v, q = _panel_vertices(case, seed)
        return dict(kind=kind, case=case, system=F.SourcePanels(v, np.zeros(len(q))),
                    external=np.random.default_rng(seed).standard_normal(len(q)))
    ev = F.Evaluation()
    if kind == "fmm":
        src, targets, vortex = _bodies(case, seed), None, _kernel(case["dist"]) == _lib.POINT_VORTEX
        kernel, potential, hessian = _kernel(case["dist"]), not vortex, vortex
    elif kind == "batch":
        counts = _batch_counts(case)
        src, targets, kernel, potential, hessian = _cube(_generator(seed), int(counts.sum())), None, _lib.POINT_SOURCE, True, False
    elif kind == "probes":
        g = _generator(seed)
        src, targets = _ring(g, case["n"], core=_core(case["n"])), _probe_points(g, case["probes"])
        kernel, potential, hessian = _lib.VORTEX_GAUSSIAN, False, False
    else:
        src, targets, kernel, potential, hessian = _panel_buffer(case, seed), None, _panel_kernel(case["shape"]), True, False
    tol = case.get("tol", 0.0)
    opt = F.make_options(expansion_order=case["p"], leaf_size_source=case["leaf"], multipole_acceptance=case["mac"],
                         error_tolerance=F.PowerRelativeGradient(tol) if tol > 0 else None, scalar_potential=potential,
                         gradient=True, hessian=hessian, precision=case.get("precision", "fp64"))
    nt = src.shape[0] if targets is None else targets.shape[0]
    return dict(kind=kind, case=case, ev=ev, opt=opt, kernel=kernel, src=src, targets=targets,
                counts=counts if kind == "batch" else None, potential=potential, hessian=hessian,
                out=torch.zeros(nt, 16, device=DEVICE, dtype=torch.float64))


# ------------------------------------------------------------------------------------------------------ passes
def _fields(out, potential, hessian):
    """The target buffer's columns as a program reads them."""
    r = {"position": out[:, :3], "gradient": out[:, 4:7]}
    if potential:
        r["potential"] = out[:, 3]
    if hessian:
        r["hessian"] = out[:, 7:16]
    return r


def run(state):
    kind, case = state["kind"], state["case"]
    if kind == "system":
        s = state["system"]
        s.reset()
        F.fmm(s, leaf_size=case["leaf"], expansion_order=case["p"], multipole_acceptance=case["mac"], hessian=True,
              evaluation=state["ev"])
        return {"velocity": s.gradient_stretching[:, :3], "gradient": s.potential[:, 4:]}
    if kind == "direct":
        s = state["system"]
        s.reset()
        F.direct(s, gradient=True, hessian=True)
        return {"velocity": s.gradient_stretching[:, :3], "gradient": s.potential[:, 4:]}
    if kind == "solve":
        s = state["system"]
        s.reset()
        solver = F.FastGaussSeidel(s, expansion_order=case["p"], multipole_acceptance=case["mac"], leaf_size=case["leaf"],
                                   influence=_lib.INFLUENCE_NORMAL_GRADIENT)
        strengths, targets, sweeps, _ = solver.solve(state["external"], max_iterations=30, tolerance=case["tol"])
        return {"strengths": strengths, "potential": targets[:, 3], "gradient": targets[:, 4:7]}
    ev = state["ev"]
    if kind == "batch":
        ev.set_batch(state["kernel"], (state["src"], state["counts"]), on_device=True)
    else:
        ev.set_systems(state["kernel"], state["targets"], state["src"], on_device=True)
    ev.fmm(state["opt"])
    return _fields(ev.targets(state["out"]), state["potential"], state["hessian"])


# -------------------------------------------------------------------------------------------------------- work
def _m2l_flops(p, vector):
    """Flops of one rotation-based multipole-to-local translation at order p."""
    h = (p + 1) * (p + 2) // 2
    f = 14 * (h - 1) + 8 * sum((n + 1) * (2 * n + 1) for n in range(p + 1)) + \
        4 * sum(p - m + 1 for n in range(p + 1) for m in range(n + 1))
    return 2 * f + 8 * h if vector else f


def work(case):
    """Bytes: each input row read and each output row written once. Flops: the body pairs and translations that the
    interaction lists of the reference hold at the acceptances used here, about 375 leaf sizes a body and 150 translations
    per leaf size of bodies (the 1M ring: 2.3e10 pairs and 1.8e6 translations; the 4M sphere: 1.0e11 and 2.3e7), at most
    half of all pairs; translations at the order an error-controlled pass mostly uses (14)."""
    kind = case["kind"]
    if kind == "solve":
        n = 6 * case["m"] ** 2
        pairs = min(100.0 * n * case["leaf"], 0.5 * n * n)
        f = pairs * 4 * 50.0 + 4 * (2.0 * pairs + 150.0 * n / case["leaf"] * _m2l_flops(case["p"], False))
        return {"bytes": 8.0 * n * (17 + 1 + 17), "flops": f}
    if kind == "direct":
        n = case["n"]
        return {"bytes": 8.0 * n * (3 + 7 + 16), "flops": 63.0 * n * n}
    rows, pair, vector = 7, 63, True
    if kind == "batch":
        n = int(_batch_counts(case).sum())
        rows, pair, vector = 5, 21, False
    elif kind == "panels":
        n = (6 if "quads" in case["shape"] else 12) * case["m"] ** 2
        rows, pair, vector = 5 + 3 * (4 if "quads" in case["shape"] else 3), 4 * 50, False
    else:
        n = case["n"]
        if case.get("dist") in ("cube", "plummer"):
            rows, pair, vector = 5, 21, False
    nt = case.get("probes", n)
    p = 14 if case.get("tol", 0.0) > 0 else case["p"]
    pairs = min((100.0 if kind == "panels" else 375.0) * nt * case["leaf"], 0.5 * nt * n)
    translations = 150.0 * max(0.0, 1.0 * nt / case["leaf"] - 4)
    return {"bytes": 8.0 * (n * rows + nt * 16 + (3 * nt if nt != n else 0)), "flops": pair * pairs + translations * _m2l_flops(p, vector)}


# ----------------------------------------------------------------------------------------------- direct sums
def _chunks(nt, ns, share=1 << 25):
    step = max(1, share // max(1, ns))
    return [(i, min(nt, i + step)) for i in range(0, nt, step)]


def _sources(t, s, q):
    """Potential and gradient slots of point sources q at s (pairs at no distance give nothing)."""
    phi, grad = torch.zeros_like(t[:, 0]), torch.zeros_like(t)
    for i, j in _chunks(len(t), len(s)):
        d = [t[i:j, None, k] - s[None, :, k] for k in range(3)]
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
        ri = torch.where(r2 > 0, torch.rsqrt(torch.where(r2 > 0, r2, torch.ones_like(r2))), torch.zeros_like(r2))
        w = q[None, :] * ri
        phi[i:j] = w.sum(1)
        w *= ri * ri
        for k in range(3):
            grad[i:j, k] = (w * d[k]).sum(1)
    f = 1.0 / (4.0 * math.pi)
    return phi * f, grad * f


def _vortex_field(t, s, gamma, sigma=None, gradient=True):
    """Velocity of point vortices gamma at s, and its derivatives d_i u_j; with sigma, of Gaussian-core vortices (velocity)."""
    u, h = torch.zeros_like(t), torch.zeros(len(t), 9, dtype=t.dtype, device=t.device)
    for i, j in _chunks(len(t), len(s)):
        d = [t[i:j, None, k] - s[None, :, k] for k in range(3)]
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
        ri = torch.where(r2 > 0, torch.rsqrt(torch.where(r2 > 0, r2, torch.ones_like(r2))), torch.zeros_like(r2))
        w3 = ri * ri * ri
        if sigma is not None:
            rho = torch.sqrt(r2) / sigma[None, :]
            w3 = w3 * (torch.erf(rho * math.sqrt(0.5)) - math.sqrt(2.0 / math.pi) * rho * torch.exp(-0.5 * rho * rho))
        # u += gamma x d / r^3, summed as moments of the weights
        c = [gamma[None, :, (k + 1) % 3] * d[(k + 2) % 3] - gamma[None, :, (k + 2) % 3] * d[(k + 1) % 3] for k in range(3)]
        for k in range(3):
            u[i:j, k] = (w3 * c[k]).sum(1)
        if gradient:
            g3 = w3 @ gamma
            w5 = -3.0 * w3 * ri * ri
            for a in range(3):
                wd = w5 * d[a]
                for b in range(3):
                    h[i:j, 3 * a + b] = (wd * c[b]).sum(1)
            # the derivative of gamma x d itself
            h[i:j, 1] += g3[:, 2]
            h[i:j, 2] -= g3[:, 1]
            h[i:j, 3] -= g3[:, 2]
            h[i:j, 5] += g3[:, 0]
            h[i:j, 6] += g3[:, 1]
            h[i:j, 7] -= g3[:, 0]
    f = 1.0 / (4.0 * math.pi)
    return u * f, h * f


def _panel_sources(t, v, c, q=None, normals=None):
    """Potential and gradient slots of constant-density planar panels v (n, nv, 3) with reference points c, by Wilton's edge sums.
    With `normals`, instead the matrix of normal gradients (targets x panels) for unit densities."""
    n, nv = v.shape[:2]
    e = v[:, 2] - v[:, 0]
    ez = torch.linalg.cross(v[:, 1] - v[:, 0], e)
    ez = ez / ez.norm(dim=1, keepdim=True)
    phi, grad = torch.zeros_like(t[:, 0]), torch.zeros_like(t)
    matrix = torch.zeros(len(t), n, dtype=t.dtype, device=t.device) if normals is not None else None
    for i, j in _chunks(len(t), n):
        d = [t[i:j, None, k] - c[None, :, k] for k in range(3)]
        z = sum(d[k] * ez[None, :, k] for k in range(3))
        z = torch.where(z == 0, torch.full_like(z, 2.0 ** -52), z)    # on the panel: its outer side
        az = z.abs()
        pot, beta = torch.zeros_like(z), torch.zeros_like(z)
        g = [torch.zeros_like(z) for _ in range(3)]
        for k in range(nv):
            a, b = v[:, k], v[:, (k + 1) % nv]
            length = (b - a).norm(dim=1)
            along = (b - a) / length[:, None]
            out = torch.linalg.cross(along, ez)
            da = [a[None, :, m] - t[i:j, None, m] for m in range(3)]
            l0 = sum(da[m] * along[None, :, m] for m in range(3))
            l1 = l0 + length[None, :]
            p = sum(da[m] * out[None, :, m] for m in range(3))
            h2 = p * p + z * z
            r0, r1 = torch.sqrt(h2 + l0 * l0), torch.sqrt(h2 + l1 * l1)
            f = torch.log((r0 + r1 + length[None, :]) / (r0 + r1 - length[None, :]))
            beta += torch.atan2(p * l1, h2 + az * r1) - torch.atan2(p * l0, h2 + az * r0)
            pot += p * f
            for m in range(3):
                g[m] += out[None, :, m] * f
        pot -= az * beta
        zb = torch.sign(z) * beta
        for m in range(3):
            g[m] += ez[None, :, m] * zb
        if normals is not None:
            matrix[i:j] = sum(normals[i:j, m, None] * g[m] for m in range(3))
        else:
            phi[i:j] = pot @ q
            for m in range(3):
                grad[i:j, m] = g[m] @ q
    f = 1.0 / (4.0 * math.pi)
    return matrix * f if normals is not None else (phi * f, grad * f)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("system", "direct"):
        if float(case["n"]) ** 2 > EXACT_PAIRS:
            return None
        b = _ring(_generator(seed), case["n"])
        u, h = _vortex_field(b[:, :3], b[:, :3], b[:, 4:7])
        return {"velocity": u, "gradient": h}
    if kind == "fmm":
        if float(case["n"]) ** 2 > EXACT_PAIRS * (0.5 if case["dist"] == "ring" else 1.0):
            return None
        b = _bodies(case, seed)
        t = b[:, :3].contiguous()
        if _kernel(case["dist"]) == _lib.POINT_VORTEX:
            u, h = _vortex_field(t, t, b[:, 4:7])
            return {"position": t, "gradient": u, "hessian": h}
        phi, grad = _sources(t, t, b[:, 4])
        return {"position": t, "gradient": grad, "potential": phi}
    if kind == "batch":
        counts = _batch_counts(case)
        b = _cube(_generator(seed), int(counts.sum()))
        parts, at = [], 0
        for n in counts.tolist():
            s = b[at:at + n]
            parts.append(_sources(s[:, :3], s[:, :3], s[:, 4]))
            at += n
        return {"position": b[:, :3], "gradient": torch.cat([x[1] for x in parts]), "potential": torch.cat([x[0] for x in parts])}
    if kind == "probes":
        g = _generator(seed)
        b, t = _ring(g, case["n"], core=_core(case["n"])), _probe_points(g, case["probes"])
        return {"position": t, "gradient": _vortex_field(t, b[:, :3], b[:, 4:7], sigma=b[:, 3], gradient=False)[0]}
    v, q = (torch.from_numpy(np.ascontiguousarray(x)).to(DEVICE) for x in _panel_vertices(case, seed))
    c = v.mean(1)
    if kind == "panels":
        if case["shape"] not in ("source_quads", "source_triangles"):
            return None
        phi, grad = _panel_sources(c, v, c, q)
        return {"position": c, "gradient": grad, "potential": phi}
    # the solve: the dense system of normal gradients, then the field of its strengths
    if len(v) > 22000:
        return None
    n = torch.linalg.cross(v[:, 1] - v[:, 0], v[:, 2] - v[:, 0])
    n = n / n.norm(dim=1, keepdim=True)
    rhs = -torch.from_numpy(np.random.default_rng(seed).standard_normal(len(v))).to(DEVICE)
    a = _panel_sources(c, v, c, normals=n)
    x = torch.linalg.solve(a, rhs)
    phi, grad = _panel_sources(c, v, c, x)
    return {"strengths": x, "potential": phi, "gradient": grad}
