"""The chunk-pruned full histogram (full_chunks.hip) against the oracle's
all-pairs loops: partly filled chunks and columns, odd and even chunk
numbers, cubic, triclinic and flat cells, open boundaries, coordinates in other
images, bins in LDS, in global memory and past the end of the array, and the
binary64 recompute with its count of re-checked pairs."""
import ctypes
import time

import numpy as np
import pytest

from fullrmc_amd import _lib, systems, tuning
from fullrmc_amd.Core import pairs_histograms as gph
from oracle import refcpu

pytestmark = pytest.mark.gpu
F32 = np.float32

CELLS = {"cubic": systems.cubic_basis(31.0), "triclinic": systems.triclinic_basis(30.0, 33.0, 36.0, 70.0, 100.0, 115.0),
         "flat": systems.triclinic_basis(60.0, 55.0, 9.0, 90.0, 80.0, 95.0), "open": None}
# nel, min, max, bin, H
GRIDS = {"lds": (2, 0.0, 9.0, 0.03, 300), "shifted": (3, 1.5, 6.0, 0.05, 90), "inter_lds": (3, 0.0, 8.0, 0.004, 2000),
         "global": (3, 0.0, 8.0, 0.0005, 16000), "past_end": (2, 0.0, 9.0, 0.03, 200), "wide": (1, 0.0, 40.0, 0.05, 800)}


def box(n, cell, seed, images):
    rng = np.random.default_rng(seed)
    f = rng.random((n, 3))
    basis = CELLS[cell] if CELLS[cell] is not None else systems.cubic_basis(31.0)
    if cell == "open":
        coords = (f * 31.0 - 7.0).astype(F32)
    else:
        coords = (f + (rng.integers(-3, 4, f.shape) if images else 0)).astype(F32)
    # a fifth of the atoms on a lattice: equal coordinates, half-cell differences
    coords[: n // 5] = (rng.integers(0, 8, (n // 5, 3)) / 8 * (31.0 if cell == "open" else 1.0)).astype(F32)
    return coords, basis, (rng.integers(0, max(1, n // 6), n)).astype(np.int32), rng


def check(n, cell, grid, images=False, f64=False, seed=0):
    nel, mn, mx, dr, H = GRIDS[grid]
    coords, basis, mol, rng = box(n, cell, seed + n, images)
    elem = rng.integers(0, nel, n).astype(np.int32)
    args = (coords, basis, cell != "open", mol, elem, nel, F32(mn), F32(mx), F32(dr), H)
    if f64:
        ri, re_, rechecked = refcpu.full_pairs_counts_f64(*args, ncores=8)
        gi, ge, _ = gph.full_pairs_histograms_coords_float64(*args)
        assert np.array_equal(gi, ri.astype(F32)) and np.array_equal(ge, re_.astype(F32))
    else:
        ri, re_ = refcpu.full_pairs_histograms_coords(*args, ncores=8)
        gi, ge = gph.full_pairs_histograms_coords(*args)
        assert gi.tobytes() == ri.tobytes() and ge.tobytes() == re_.tobytes()
    return gi.sum() + ge.sum()


@pytest.mark.parametrize("cell", sorted(CELLS))
@pytest.mark.parametrize("n", [95, 192, 577, 1409, 4096, 4097, 9001])
def test_sizes_and_cells(n, cell):
    assert check(n, cell, "lds") > 0
    assert check(n, cell, "shifted", images=True) > 0


@pytest.mark.parametrize("n", [2, 3, 13, 63, 64, 65, 128])
def test_smallest(n):
    for cell in sorted(CELLS):
        check(n, cell, "wide", images=cell != "open", seed=40)
        check(n, cell, "wide", f64=True, seed=41)


@pytest.mark.parametrize("grid", sorted(GRIDS))
@pytest.mark.parametrize("cell", ["cubic", "triclinic", "open"])
def test_grids(grid, cell):
    assert check(2000, cell, grid, seed=5) > 0


@pytest.mark.parametrize("cell", sorted(CELLS))
@pytest.mark.parametrize("grid", ["lds", "shifted", "inter_lds", "wide"])
def test_binary64(grid, cell):
    assert check(1500, cell, grid, images=cell != "open", f64=True, seed=9) > 0


def test_all_pairs_and_chunks_give_the_same_recheck_count():
    coords, basis, mol, rng = box(3000, "triclinic", 3, True)
    elem = rng.integers(0, 2, 3000).astype(np.int32)
    args = (coords, basis, True, mol, elem, 2, F32(0.0), F32(9.0), F32(0.01), 900)
    a = gph.full_pairs_histograms_coords_float64(*args)
    tuning.force_full_schedule(256, 2, 2)
    try:
        b = gph.full_pairs_histograms_coords_float64(*args)
    finally:
        tuning.force_full_schedule()
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]) and a[2] == b[2] > 0


def test_coordinates_that_are_not_finite_are_never_in_range():
    coords, basis, mol, rng = box(900, "cubic", 4, False)
    coords[17], coords[400, 1], coords[800, 2] = np.nan, np.inf, -np.inf
    elem = rng.integers(0, 2, 900).astype(np.int32)
    grid = (2, F32(0.0), F32(9.0), F32(0.03), 300)
    got = gph.full_pairs_histograms_coords(coords, basis, True, mol, elem, *grid)
    keep = np.all(np.isfinite(coords), axis=1)
    want = refcpu.full_pairs_histograms_coords(coords[keep], basis, True, mol[keep], elem[keep], *grid, ncores=8)
    assert got[0].tobytes() == want[0].tobytes() and got[1].tobytes() == want[1].tobytes()


def test_kernel_time_holds_no_wait_for_the_host():
    """frmc_last_kernel_ms covers the pass alone, so it is not above the whole call's
    time without timing; the evaluated pairs are counted all the same."""
    import torch
    rng = np.random.default_rng(6)
    n, H, L = 13500, 1000, _lib.lib()
    dev = [torch.from_numpy(a).cuda() for a in
           (rng.random((n, 3), F32), np.diag([45.0, 45.0, 90.0]).astype(F32), np.arange(n, dtype=np.int32) // 3,
            rng.integers(0, 2, n).astype(np.int32), np.zeros((2, 2, 2, H), F32))]
    c, b, m, e, out = (t.data_ptr() for t in dev)

    def call():
        t0 = time.perf_counter()
        _lib.check(L.frmc_full_pairs_histograms_coords(c, n, b, 1, m, e, 2, 0.0, 20.0, 0.02, H, out, out + 16 * H,
                                                       torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        return time.perf_counter() - t0

    whole = min(call() for _ in range(20))
    evaluated = ctypes.c_int64(0)
    L.frmc_set_timing(1)
    try:
        kernel = []
        for _ in range(20):
            call()
            kernel.append(L.frmc_last_kernel_ms() * 1e-3)
        _lib.check(L.frmc_last_full_evaluated(ctypes.byref(evaluated)))
    finally:
        L.frmc_set_timing(0)
    counted = int(dev[4].sum().item())
    assert counted <= evaluated.value <= n * n
    assert min(kernel) < 1.3 * whole, (min(kernel), whole)


@pytest.mark.parametrize("n", [100, 1000, 4096])
def test_few_atoms_of_many_elements(n):
    """Up to 64 elements of 1,000 bins: the counts are cleared and converted by the
    whole chip (in the one workgroup that sorts few atoms: ten times the time of 2
    elements at 1,000 atoms, now 2.3 times)."""
    import torch
    coords, basis, mol, rng = box(n, "triclinic", 8, True)
    grid = (F32(0.0), F32(9.0), F32(0.009), 1000)
    best = {}
    for nel in (2, 6, 64):
        elem = rng.integers(0, nel, n).astype(np.int32)
        ri, re_ = refcpu.full_pairs_histograms_coords(coords, basis, True, mol, elem, nel, *grid, ncores=8)
        gi, ge = gph.full_pairs_histograms_coords(coords, basis, True, mol, elem, nel, *grid)
        assert gi.tobytes() == ri.tobytes() and ge.tobytes() == re_.tobytes()
        dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (coords, basis, mol, elem)]
        out = torch.empty((2, nel, nel, 1000), device="cuda")
        c, b, m, e = (t.data_ptr() for t in dev)
        times = []
        for _ in range(12):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            _lib.check(_lib.lib().frmc_full_pairs_histograms_coords(
                c, n, b, 1, m, e, nel, *grid, out[0].data_ptr(), out[1].data_ptr(),
                torch.cuda.current_stream().cuda_stream))
            times.append(time.perf_counter() - t0)
        best[nel] = min(times)
    assert best[64] < 5 * best[2], best


@pytest.mark.parametrize("n", [4097, 9001])
@pytest.mark.parametrize("case", ["far", "offset", "line", "point", "not finite", "two clusters"])
def test_open_boundaries_of_uneven_extent(n, case):
    """Open boundaries whose extent says little about where the atoms are: the sort's
    cells cover the bulk of them, the rest fall into the cells at the ends."""
    rng = np.random.default_rng(n)
    coords = rng.random((n, 3)) * 40.0
    if case == "far":
        coords[5] = 1e7, -3e5, 2e4
    elif case == "offset":
        coords += 5000.0
    elif case == "line":
        coords[:, 1:] = 3.0
    elif case == "point":
        coords[:] = 1.5
        coords[: n // 2] += 6.0
    elif case == "not finite":
        coords[7, 0], coords[80, 1], coords[900, 2] = np.nan, np.inf, 2e38
    else:
        coords[n // 3:] += 3e4
    coords = coords.astype(F32)
    mol, elem = (np.arange(n) // 3).astype(np.int32), rng.integers(0, 2, n).astype(np.int32)
    grid = (2, F32(0.0), F32(9.0), F32(0.03), 300)
    basis = systems.cubic_basis(40.0)
    got = gph.full_pairs_histograms_coords(coords, basis, False, mol, elem, *grid)
    keep = np.all(np.isfinite(coords), axis=1)
    want = refcpu.full_pairs_histograms_coords(coords[keep], basis, False, mol[keep], elem[keep], *grid, ncores=8)
    assert got[0].sum() + got[1].sum() > 0
    assert got[0].tobytes() == want[0].tobytes() and got[1].tobytes() == want[1].tobytes()


def test_one_atom_far_away_costs_no_more_than_all_pairs():
    """50,000 atoms in open boundaries and one of them at a thousand times their extent:
    436 us a call, 1,312 when the extent alone gave the cells, all pairs 874."""
    import torch
    rng = np.random.default_rng(3)
    n, H, side = 50000, 600, 91.0
    coords = (rng.random((n, 3)) * side).astype(F32)
    coords[0] = 1000 * side
    dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in
           (coords, systems.cubic_basis(side), np.arange(n, dtype=np.int32) // 3, rng.integers(0, 2, n).astype(np.int32),
            np.zeros((2, 2, 2, H), F32))]
    c, b, m, e, out = (t.data_ptr() for t in dev)
    best = {}
    for on in (True, False):
        tuning.set_autotune(on)
        try:
            times = []
            for _ in range(6):
                torch.cuda.synchronize()
                t0 = time.perf_counter()
                _lib.check(_lib.lib().frmc_full_pairs_histograms_coords(
                    c, n, b, 0, m, e, 2, 0.0, 12.0, 0.02, H, out, out + 16 * H, torch.cuda.current_stream().cuda_stream))
                torch.cuda.synchronize()
                times.append(time.perf_counter() - t0)
            best[on] = min(times)
        finally:
            tuning.set_autotune(True)
    assert best[True] < 0.8 * best[False], best
