"""Distances at the ends of the FP64 point source's two reciprocal-root paths with a potential (normal floats of r^2, and
the rest), and the one path without.

A nearfield-only evaluation (one leaf) of bodies whose spacing spans r^2 across the FP32 range's lower and upper ends,
with coincident bodies, against the same sums in extended precision. Each pair is accurate to about two units in the
last place, so 1e-14 of the sum of the pairs' magnitudes."""
import numpy as np
import pytest

import fastmultipole_amd as F
from fastmultipole_amd import _lib


def check(n, scale, potential=True, gradient=True):
    rng = np.random.default_rng(5)
    b = np.zeros((n, 5))
    b[:, :3] = rng.normal(size=(n, 3))
    c, m = min(10, n // 7), 4 * n // 7
    b[m:m + c, :3] = b[:c, :3]                          # coincident bodies
    b[m + c:m + 2 * c, :3] = b[c:2 * c, :3] + 1e-3 * rng.normal(size=(c, 3))
    b[:, :3] *= scale
    b[:, 4] = rng.normal(size=n)
    ev = F.Evaluation()
    ev.set_systems(_lib.POINT_SOURCE, None, b)
    ev.fmm(F.make_options(expansion_order=4, leaf_size_source=100, scalar_potential=potential, gradient=gradient))
    out = ev.targets()
    ev.close()
    x = b[:, :3].astype(np.longdouble)
    d = x[:, None] - x[None]
    r2 = (d ** 2).sum(2)
    ri = np.where(r2 > 0, 1 / np.sqrt(np.where(r2 > 0, r2, 1)), 0)
    q = b[:, 4].astype(np.longdouble) / (4 * np.longdouble(np.pi))
    phi, grad = q[None] * ri, (q[None] * ri ** 3)[..., None] * d
    if potential:
        assert np.abs(out[:, 3] - phi.sum(1).astype(float)).max() <= 1e-14 * np.abs(phi).sum(1).max()
    if gradient:
        assert np.abs(out[:, 4:7] - grad.sum(1).astype(float)).max() <= 1e-14 * np.abs(grad).sum(1).max()


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [1.0, 1e-17, 1e-19, 3e-20, 1e-30, 1e18, 3e19, 1e25])
def test_point_source_pairs_at_every_scale(scale):
    check(70, scale)


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [1.0, 1e-19])
@pytest.mark.parametrize("n", [7, 14, 33, 64, 71, 99, 100])
@pytest.mark.parametrize("switches", [(True, True), (True, False), (False, True)], ids=["both", "potential", "gradient"])
def test_leaves_of_every_share_of_sources(n, switches, scale):
    """Leaves whose sources leave the lanes a rest or none, with and without the potential."""
    check(n, scale, *switches)
