"""The panel nearfield's closed form at targets where its terms degenerate: centroids (on the panel, on a quadrilateral's
diagonal), points 1e-3 off edge midpoints and vertices, points a hair off a panel's plane, far points; and, in tests of
their own, targets exactly on edges and at vertices. direct! of
every panel on every such target, to 1e-10 of the largest value of a quantity: what the solid angle
enters (source panels' potential and gradient, dipole panels' potential) against the edge sums of Wilton et al. (1984) in
extended precision, the rest against the oracle's reference form. (At triangles of size 1e-7 the reference's arctangents at
a centroid, moved off the plane by eps(), are 1.9e-10 off.)"""
import numpy as np
import pytest

import fastmultipole_amd as F
from fastmultipole_amd import _lib, workloads as W
from oracle import oracle as O

KINDS = {"source-quads": (_lib.PANEL_SOURCE_QUAD, 6), "source-triangles": (_lib.PANEL_SOURCE_TRI, 4),
         "dipole-quads": (_lib.PANEL_DIPOLE_QUAD, 7), "dipole-triangles": (_lib.PANEL_DIPOLE_TRI, 5)}


def edge_sums(t, v, c):
    """Potential and gradient slots of unit source panels v (n, nv, 3) with reference points c at t, and the potential slot of
    unit dipole panels, summed, in long double."""
    t, v, c = (np.asarray(x, dtype=np.longdouble) for x in (t, v, c))
    e = v[:, 2] - v[:, 0]
    ez = np.cross(v[:, 1] - v[:, 0], e)
    ez /= np.sqrt((ez ** 2).sum(1))[:, None]
    z = ((t[:, None] - c[None]) * ez[None]).sum(2)
    z = np.where(z == 0, np.longdouble(2.0) ** -52, z)   # on the panel: its outer side
    az = abs(z)
    phi, beta, g = 0, 0, 0
    for k in range(v.shape[1]):
        a, b = v[:, k], v[:, (k + 1) % v.shape[1]]
        length = np.sqrt(((b - a) ** 2).sum(1))
        along = (b - a) / length[:, None]
        out = np.cross(along, ez)
        d = a[None] - t[:, None]
        l0, p = (d * along[None]).sum(2), (d * out[None]).sum(2)
        l1, h = l0 + length, p * p + z * z
        r0, r1 = np.sqrt(h + l0 * l0), np.sqrt(h + l1 * l1)
        # on an edge the difference rounds to zero or below it: p f is then below any rounding of phi
        f = np.log1p(2 * length / np.maximum(r0 + r1 - length, np.longdouble(2.0) ** -100))
        beta = beta + np.arctan2(p * l1, h + az * r1) - np.arctan2(p * l0, h + az * r0)
        phi, g = phi + p * f, g + out[None] * f[..., None]
    g = g + ez[None] * (np.sign(z) * beta)[..., None]
    f4 = 1 / (4 * np.longdouble(np.pi))
    return [(x.sum(1) * f4).astype(float) for x in (phi - az * beta, g, np.sign(z) * beta)]


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [1.0, 1e-6, 1e5])
@pytest.mark.parametrize("name", list(KINDS))
def test_direct_at_degenerate_targets(name, scale):
    kernel, okind = KINDS[name]
    rows, _ = W.sphere_panels(3, quads="quads" in name, seed=9)
    rows[:, 4] = 1.0
    if "quads" in name:   # squares in one plane: symmetric panels, whose edge angles at the centroid are right angles
        sq = np.array([[[i, j, 3.0], [i + 1, j, 3.0], [i + 1, j + 1, 3.0], [i, j + 1, 3.0]] for i in range(2) for j in range(2)])
        rows = np.concatenate([rows, W.panel_rows(sq, np.ones(4))])
    v = rows[:, 5:].reshape(len(rows), -1, 3)
    rng = np.random.default_rng(1)
    n = v[:, 1] - v[:, 0]
    n = np.cross(n, v[:, 2] - v[:, 0])
    n /= np.linalg.norm(n, axis=1)[:, None]
    off = np.exp(rng.uniform(np.log(1e-7), np.log(1.0), len(v)))[:, None]
    t = np.concatenate([rows[:, :3], rows[:, :3] + off * n, rows[:, :3] - off * n,
                        0.5 * (v[:, 0] + v[:, 1]) + 1e-3 * n, v[:, 2] - 1e-3 * n, 20.0 * rng.normal(size=(8, 3))])
    rows = rows.copy()
    rows[:, :4] *= scale
    rows[:, 5:] *= scale
    t = np.ascontiguousarray(t * scale)
    out = np.zeros((len(t), 16))
    ctx = F.default_context()
    rows = np.ascontiguousarray(rows)
    hess = "dipole" not in name   # a dipole panel's Hessian is not defined on its own plane
    ctx.check(ctx.lib.fmmhip_direct(ctx._h, kernel, len(t), t.ctypes.data, len(rows), rows.ctypes.data, 1, 1, int(hess),
                                    _lib.FP64, out.ctypes.data, 0))
    ref = O.direct(okind, t, rows, True, True, hess)
    phi, grad, dipole = edge_sums(t, rows[:, 5:].reshape(len(rows), -1, 3), rows[:, :3])
    if "source" in name:
        ref[:, 3], ref[:, 4:7] = phi, grad
    else:
        ref[:, 3] = dipole
    for lo, hi in ((3, 4), (4, 7)) + (((7, 16),) if hess else ()):
        assert np.isfinite(out[:, lo:hi]).all()
        assert np.abs(out[:, lo:hi] - ref[:, lo:hi]).max() <= 1e-10 * np.abs(ref[:, lo:hi]).max(), (lo, hi)


def direct(kernel, rows, t, hessian=False):
    """direct! of every panel row on every target: potential, gradient (and Hessian) slots."""
    rows, t = np.ascontiguousarray(rows), np.ascontiguousarray(t)
    out = np.zeros((len(t), 16))
    ctx = F.default_context()
    ctx.check(ctx.lib.fmmhip_direct(ctx._h, kernel, len(t), t.ctypes.data, len(rows), rows.ctypes.data, 1, 1, int(hessian),
                                    _lib.FP64, out.ctypes.data, 0))
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [1.0, 1e-6, 1e5])
@pytest.mark.parametrize("name", ["source-quads", "source-triangles", "source-dipole-quads", "source-dipole-triangles"])
def test_targets_on_edges_and_at_vertices(name, scale):
    """Targets exactly on panels' edges (midpoints, other fractions) and at their vertices, where the sum of the distances to
    an edge's ends rounds to its length or below it. The potential is finite there: against the edge sums in extended
    precision. The gradient is logarithmically infinite: each edge's logarithm is at most the one of the reference's eps()
    perturbation, |log(eps() / 2d)| < 60 at these scales."""
    rows, _ = W.sphere_panels(5, quads="quads" in name, seed=4)
    rows[:, 4] = 1.0
    v = rows[:, 5:].reshape(len(rows), -1, 3)
    nv = v.shape[1]
    rng = np.random.default_rng(2)
    edge = rng.integers(0, nv, len(v))
    a, b = v[np.arange(len(v)), edge], v[np.arange(len(v)), (edge + 1) % nv]
    s = rng.uniform(0.0, 1.0, len(v))[:, None]
    t = np.concatenate([0.5 * (a + b), a + s * (b - a), a]) * scale
    rows = rows.copy()
    rows[:, :4] *= scale
    rows[:, 5:] *= scale
    phi, _, _ = edge_sums(t, rows[:, 5:].reshape(len(rows), -1, 3), rows[:, :3])
    if "dipole" in name:   # no dipole strength: the source's potential and gradient
        kernel = _lib.PANEL_SOURCE_DIPOLE_QUAD if nv == 4 else _lib.PANEL_SOURCE_DIPOLE_TRI
        out = direct(kernel, np.insert(rows, 5, 0.0, axis=1), t)
    else:
        out = direct(KINDS[name][0], rows, t)
        assert np.isfinite(out[:, 4:7]).all()
        assert np.abs(out[:, 4:7]).max() < len(v) * nv * 60 / (4 * np.pi)
    assert np.isfinite(out[:, 3]).all()
    assert np.abs(out[:, 3] - phi).max() <= 1e-10 * np.abs(phi).max()


@pytest.mark.gpu
@pytest.mark.parametrize("distance", [1.0, 1e3, 3e4])
@pytest.mark.parametrize("name", ["source-quads", "dipole-quads"])
def test_sliver_edges_seen_from_afar(name, distance):
    """Pole quadrilaterals of a sphere meshed in latitude and longitude: the first edge is sin(pi) = 1.2e-16 of the radius
    wide, up to 1e21 times shorter than the distance. The solid angle's eight edge ends each carry a rounding of at most
    8 2^-53 of a right angle's tangent, 32 2^-52 in all; the rest of a value is good to 1e-13."""
    n, polar = 20, np.array([np.pi, np.pi - 0.1])
    phi = np.linspace(0.0, 2 * np.pi, n + 1)
    point = lambda th, ph: np.stack([np.sin(th) * np.cos(ph), np.sin(th) * np.sin(ph), np.cos(th) + 0 * ph], axis=-1)
    lo, hi = point(polar[0], phi), point(polar[1], phi)
    rows = W.panel_rows(np.stack([lo[:-1], lo[1:], hi[1:], hi[:-1]], axis=1), np.ones(n))
    t = np.random.default_rng(6).normal(size=(40, 3))
    t *= distance / np.linalg.norm(t, axis=1)[:, None]
    out = direct(KINDS[name][0], rows, t)
    ref, grad, dipole = edge_sums(t, rows[:, 5:].reshape(n, 4, 3), rows[:, :3])
    angle = n * 32 * 2.0 ** -52 / (4 * np.pi)
    assert np.isfinite(out[:, 3:7]).all()
    if name == "dipole-quads":
        assert np.abs(out[:, 3] - dipole).max() <= angle
    else:
        assert np.abs(out[:, 3] - ref).max() <= 1e-13 * np.abs(ref).max() + angle * 1.1 * distance
        assert np.abs(out[:, 4:7] - grad).max() <= 1e-13 * np.abs(grad).max() + angle


@pytest.mark.gpu
@pytest.mark.parametrize("repeat", [[0, 1, 2, 2], [0, 1, 2, 0]], ids=["third-vertex-twice", "first-vertex-twice"])
@pytest.mark.parametrize("name", ["source", "dipole", "source-dipole"])
def test_quadrilaterals_with_a_repeated_vertex(name, repeat):
    """Triangles handed over as quadrilaterals with a vertex given twice: the edge of no length adds nothing, so every output
    is the triangle kernel's up to rounding (1e-12 of the largest value)."""
    kinds = {"source": (_lib.PANEL_SOURCE_TRI, _lib.PANEL_SOURCE_QUAD), "dipole": (_lib.PANEL_DIPOLE_TRI, _lib.PANEL_DIPOLE_QUAD),
             "source-dipole": (_lib.PANEL_SOURCE_DIPOLE_TRI, _lib.PANEL_SOURCE_DIPOLE_QUAD)}[name]
    rows = W.sphere_source_dipole_panels(3, quads=False, seed=3)[0]
    if "-" not in name:
        rows = np.delete(rows, 5, axis=1)
    at = rows.shape[1] - 9
    v = rows[:, at:].reshape(-1, 3, 3)
    quads = np.concatenate([rows[:, :at], v[:, repeat].reshape(len(v), 12)], axis=1)
    rng = np.random.default_rng(8)
    t = np.concatenate([rng.normal(size=(40, 3)), 0.2 * rng.normal(size=(10, 3))])
    tri, quad = (direct(k, r, t, hessian=True) for k, r in zip(kinds, (rows, quads)))
    for lo, hi in ((3, 4), (4, 7), (7, 16)):
        assert np.abs(quad[:, lo:hi] - tri[:, lo:hi]).max() <= 1e-12 * np.abs(tri[:, lo:hi]).max(), (lo, hi)
