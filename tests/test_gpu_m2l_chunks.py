"""Chunks of long M2L lists in the matrix-core engine (m2l_mx_gpu.hpp).

Target boxes whose lists are shorter than, equal to and longer than one chunk, at every order cap, against the
wavefront engine (one wavefront per interaction, no chunks). Both apply the same operators to the same lists; only
the order of the sums differs, so the outputs agree to 1e-11 relative, the bar the library's engines are held to."""
import numpy as np
import pytest

import fastmultipole_amd as F
from fastmultipole_amd import _lib, workloads as W

CHUNK = {8: 8, 12: 8, 16: 16, 20: 16}   # vortex interactions per chunk at each order cap; twice as many of one potential


@pytest.mark.parametrize("S", [8, 16, 32])
def test_slots_of_boxes_never_overlap(S):
    """Box b's chunks take slots l0 // S + b + c: disjoint between boxes, below n // S + n_boxes."""
    lens = np.array([1, S - 1, S, S + 1, 2 * S, 2 * S + 1, 1, 7 * S, 3, S, S, 5 * S - 1])
    off = np.concatenate([[0], np.cumsum(lens)])
    slots = np.concatenate([off[b] // S + b + np.arange(-(-n // S)) for b, n in enumerate(lens)])
    assert len(np.unique(slots)) == len(slots)
    assert slots.max() < off[-1] // S + len(lens)


@pytest.mark.gpu
@pytest.mark.parametrize("kernel", [_lib.POINT_SOURCE, _lib.POINT_VORTEX], ids=["source", "vortex"])
@pytest.mark.parametrize("p", [7, 8, 12, 15, 20])
def test_chunked_lists_match_the_wavefront_engine(p, kernel, monkeypatch):
    rows = W.plummer_sources(2600, seed=11) if kernel == _lib.POINT_SOURCE else W.uniform_vortices(2600, seed=11)
    S = CHUNK[min(c for c in CHUNK if c >= p)] * (1 if kernel == _lib.POINT_VORTEX else 2)
    outs = {}
    for engine in ("mx", "wave"):
        monkeypatch.setenv("FMMHIP_M2L_KERNEL", engine)
        ev = F.Evaluation()
        ev.set_systems(kernel, None, rows)
        ev.fmm(F.make_options(expansion_order=p, leaf_size_source=12, multipole_acceptance=0.6, scalar_potential=True,
                              gradient=True, hessian=True))
        outs[engine] = ev.targets()
        lens = np.bincount(ev.list(0)[:, 0])
        ev.close()
    lens = lens[lens > 0]
    assert lens.max() > 2 * S and lens.min() < S
    for lo, hi in ((3, 4), (4, 7), (7, 16)):
        ref = outs["wave"][:, lo:hi]
        assert np.abs(outs["mx"][:, lo:hi] - ref).max() <= 1e-11 * max(np.abs(ref).max(), 1e-300)
