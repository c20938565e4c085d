"""Chunks of long M2L lists in the matrix-core engine (m2l_mx_gpu.hpp).

Target boxes whose lists are shorter than, equal to and longer than one chunk, at every order cap, against the
wavefront engine (one wavefront per interaction, no chunks). Both apply the same operators to the same lists; only
the order of the sums differs, so the outputs agree to 1e-11 relative, the bar the library's engines are held to."""
import ctypes

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


@pytest.mark.parametrize("S,n_branches,room", [(8, 40, 12), (16, 700, 100), (32, 33, 5), (8, 1000, 251)])
def test_passes_take_every_box_once_and_stay_in_the_workspace(S, n_branches, room):
    """Passes of room - span slots, span the chunks of the longest list possible: each box's chunks lie in one pass, at
    workspace slots below room."""
    rng = np.random.default_rng(S)
    lens = np.concatenate([rng.integers(1, n_branches + 1, 300), np.full(5, n_branches), np.full(40, 1)])
    off = np.concatenate([[0], np.cumsum(lens)])
    first = off[:-1] // S + np.arange(len(lens))
    chunks = -(-lens // S)
    slots, span = off[-1] // S + len(lens), -(-n_branches // S)
    room = max(room, 2 * span)
    taken = np.zeros(len(lens), int)
    for w0 in range(0, slots, room - span):
        w1 = min(slots, w0 + room - span)
        mine = (first >= w0) & (first < w1)
        taken += mine
        assert (first + chunks)[mine].max(initial=0) <= min(slots, w1 + span)
        assert (first + chunks - w0)[mine].max(initial=0) <= room
    assert (taken == 1).all()


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


@pytest.mark.gpu
@pytest.mark.parametrize("kernel", [_lib.POINT_SOURCE, _lib.POINT_VORTEX], ids=["source", "vortex"])
@pytest.mark.parametrize("p,tol", [(8, 1e-3), (12, 1e-5), (16, 1e-6), (20, 1e-8)])
def test_chunked_error_controlled_lists_match_the_wavefront_engine(p, tol, kernel, monkeypatch):
    """Orders chosen per interaction, lists longer than a chunk, processed in an order of their own. The engines' test values
    agree to a few ulps, so every order is the same (a tolerance within an ulp's reach of one is not met by 1e5 tests)."""
    rows = W.plummer_sources(2600, seed=11) if kernel == _lib.POINT_SOURCE else W.uniform_vortices(2600, seed=11)
    S = CHUNK[min(c for c in CHUNK if c >= p)] * (1 if kernel == _lib.POINT_VORTEX else 2)
    outs, orders = {}, {}
    for engine in ("mx", "wave"):
        monkeypatch.setenv("FMMHIP_M2L_KERNEL", engine)
        ev = F.Evaluation()
        ev.set_systems(kernel, None, rows)
        ev.fmm(F.make_options(expansion_order=p, leaf_size_source=12, multipole_acceptance=0.6, scalar_potential=True,
                              gradient=True, hessian=True, error_tolerance=F.PowerRelativeGradient(tol)))
        outs[engine], orders[engine] = ev.targets(), ev.m2l_orders()
        lens = np.bincount(ev.list(0)[:, 0])
        ev.close()
    assert lens.max() > 2 * S
    np.testing.assert_array_equal(orders["mx"], orders["wave"])
    assert len(np.unique(orders["mx"])) > 2
    for lo, hi in ((3, 4), (4, 7), (7, 16)):
        ref = outs["wave"][:, lo:hi]
        assert np.abs(outs["mx"][:, lo:hi] - ref).max() <= 1e-11 * max(np.abs(ref).max(), 1e-300)


def _free_bytes():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert _lib.load().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0   # the runtime the library is linked to
    return free.value


@pytest.mark.gpu
def test_partial_expansions_take_a_bounded_workspace(monkeypatch):
    """Lists of 37M interactions whose partial expansions would take 19 GB: the workspace is at most 2 GiB (and the buffers'
    eighth of slack), boxes are taken in passes. Outputs against the wavefront engine, and a system evaluated beside
    the large one (in the last pass) bit for bit as by itself."""
    big, small = W.uniform_vortices(2500000, seed=5), W.uniform_vortices(20000, seed=6)
    opt = F.make_options(expansion_order=20, leaf_size_source=20, multipole_acceptance=0.5, gradient=True)
    outs = {}
    ev = F.Evaluation()
    ev.set_batch(_lib.POINT_VORTEX, [big, small])
    for engine in ("wave", "mx"):   # the same handle: all other buffers have their size after the first
        monkeypatch.setenv("FMMHIP_M2L_KERNEL", engine)
        before = _free_bytes()
        s = ev.fmm(opt)
        grown = before - _free_bytes()
        outs[engine] = ev.targets()[:, 4:7]
        print(f"{engine}: {s.n_m2l} interactions, {s.ms_m2l:.1f} ms, grown by {grown / 2**20:.0f} MiB", flush=True)
    ev.close()
    assert s.n_m2l // CHUNK[20] * 4 * 231 * 8 > 4 * 2**30
    assert grown < 2.3 * 2**30
    assert np.abs(outs["mx"] - outs["wave"]).max() <= 1e-11 * np.abs(outs["wave"]).max()
    alone = F.Evaluation()
    alone.set_systems(_lib.POINT_VORTEX, None, small)
    alone.fmm(opt)
    np.testing.assert_array_equal(alone.targets()[:, 4:7], outs["mx"][len(big):])
    alone.close()
