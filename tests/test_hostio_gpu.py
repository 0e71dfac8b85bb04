"""Bulk data between host arrays and the device in pinned chunks: score reads,
segmentation and dose table of host arrays, at sizes around one chunk, one
round of slots and many of them, and from several threads at once."""
from __future__ import annotations

from concurrent.futures import ThreadPoolExecutor

import ctypes as C
import subprocess
import threading

import numpy as np
import pytest

import opendxmc_amd as dx
from opendxmc_amd import _native as N
from opendxmc_amd import build
from opendxmc_amd import phantoms
from opendxmc_amd import pipelines as P
from opendxmc_amd.devmem import DeviceBuffer, _rt
from physics_refs import MGY_PER_KEV_G

pytestmark = pytest.mark.gpu


def scored_world(dims, histories=200_000, seed=3):
    n = int(np.prod(dims))
    rng = np.random.default_rng(seed)
    density = rng.uniform(0.5, 1.5, n)
    density[rng.random(n) < 0.02] = 0.0     # no mass: dose 0 whatever was scored
    world = dx.World()
    grid = world.addItem(dx.AAVoxelGrid(correction=0))
    grid.setData(dims, density, np.ones(n, dtype=np.uint8), [dx.Material.byWeight(m) for m in (phantoms.AIR, phantoms.WATER)])
    grid.setSpacing((0.1, 0.1, 0.1))
    world.build()
    beam = dx.DXBeam({13: 2.0})
    beam.setCollimation((2.0, 2.0))
    beam.setNumberOfParticlesPerExposure(histories)
    assert dx.Transport(seed=seed)(world, beam, None, False)
    return world, grid, density


# voxels per chunk: 16,448 at least and 131,072 at most, 16 slots, 12 threads
@pytest.mark.parametrize("dims", [(3, 1, 1), (64, 257, 1), (16449, 1, 1), (101, 97, 43), (131073, 2, 1), (128, 128, 130), (200, 181, 120)])
def test_scores_read_whole(dims):
    world, grid, density = scored_world(dims)
    e, e2, ev = grid.energyScored()
    c = grid.counters()
    assert int(ev.sum()) == c["deposits"]
    # FP64 sums of the same FP32 deposits in another order
    np.testing.assert_allclose(e.sum(), c["deposited_energy"], rtol=1e-10)
    assert ((ev > 0) == (e > 0)).all() and (e2 <= e * e * (1 + 1e-12)).all()
    dose, var, ev2 = grid.doseScored()
    np.testing.assert_array_equal(ev2, ev)
    h = float(grid.histories())
    mass = density * 1e-3    # g in 0.1 cm voxels
    with np.errstate(divide="ignore", invalid="ignore"):
        f = np.where(mass > 0, MGY_PER_KEV_G / mass, 0.0)
    np.testing.assert_allclose(dose, e * f, rtol=1e-12)
    np.testing.assert_allclose(var, np.maximum(0.0, h / (h - 1) * (e2 - e * e / h)) * f * f, rtol=1e-9)
    # the arrays one at a time: the others null
    for k in range(3):
        out = [np.full(grid.size(), 7, dtype=t) for t in (np.float64, np.float64, np.uint64)]
        ptrs = [N.ptr(out[0], C.c_double), N.ptr(out[1], C.c_double), N.ptr(out[2], N.u64)]
        N.check(N.lib().dxg_read_dose_scores(grid._h, *[p if i == k else None for i, p in enumerate(ptrs)]))
        np.testing.assert_array_equal(out[k], (dose, var, ev)[k])
        N.check(N.lib().dxg_read_energy_scores(grid._h, *[p if i == k else None for i, p in enumerate(ptrs)]))
        np.testing.assert_array_equal(out[k], (e, e2, ev)[k])
        assert all((out[i] == 7).all() for i in range(3) if i != k)


@pytest.mark.parametrize("dims", [(16, 16, 16), (101, 97, 43)])
def test_read_after_an_unrelated_error(dims):
    """An error that an earlier call of the runtime left behind on the thread is
    not taken for the read's own."""
    _, grid, _ = scored_world(dims)
    want = grid.doseScored()
    assert _rt().hipSetDevice(9999) != 0
    try:
        for a, b in zip(grid.doseScored(), want):
            np.testing.assert_array_equal(a, b)
        assert _rt().hipPeekAtLastError() != 0      # still its owner's to find
    finally:
        _rt().hipGetLastError()


def test_concurrent_reads():
    """More readers than kept slot sets, on worlds of different sizes."""
    worlds = [scored_world(d, seed=s) for s, d in enumerate([(101, 97, 43), (128, 128, 130), (60, 60, 60), (200, 181, 40)])]
    want = [g.doseScored() for _, g, _ in worlds]
    jobs = [k % 4 for k in range(16)]
    with ThreadPoolExecutor(8) as pool:
        got = list(pool.map(lambda k: worlds[k][1].doseScored(), jobs))
    for k, r in zip(jobs, got):
        for a, b in zip(r, want[k]):
            np.testing.assert_array_equal(a, b)


def test_read_during_runs_is_a_state_between_launches():
    """Events read in one thread while another runs one launch after the other:
    every read is the scores after some launch, none a mixture of several."""
    world, grid, _ = scored_world((200, 181, 120), histories=20_000)   # one tally copy, 23 chunks a read
    beam = dx.DXBeam({13: 2.0})
    beam.setCollimation((20.0, 20.0))
    beam.setNumberOfParticlesPerExposure(200_000)
    states, stop = [grid.counters()["deposits"]], threading.Event()

    def run():
        tr = dx.Transport(seed=9)
        for _ in range(2000):
            if stop.is_set() or not tr(world, beam, None, False):
                break
            states.append(states[-1] + grid.counters()["deposits"])

    thread = threading.Thread(target=run)
    thread.start()
    try:
        reads = []
        for _ in range(12):
            ev = np.empty(grid.size(), dtype=np.uint64)
            N.check(N.lib().dxg_read_energy_scores(grid._h, None, None, N.ptr(ev, N.u64)))
            reads.append(int(ev.sum()))
    finally:
        stop.set()
        thread.join()
    assert reads[0] < reads[-1]
    assert set(reads) <= set(states)


@pytest.mark.parametrize("n", [1, 393_215, 393_216, (1 << 19) - 1, 1 << 19, 12 * 23168 + 1, 16 * 185024 + 5, 4_000_037])
def test_segmentation_of_host_arrays_equals_resident(n):
    """The same bits whichever way the voxels travel, below 393,216 voxels through
    whole device buffers and from there in chunks; with the densities over the CT
    numbers too, and over the materials."""
    rng = np.random.default_rng(n)
    hu = rng.uniform(-1100.0, 2500.0, n)
    hu[rng.integers(0, n, 5)] = [np.nan, np.inf, -np.inf, -0.0, -1000.0]
    tables = P.CTSegmentationPipeline().tables()
    bufs = [DeviceBuffer.from_array(hu), DeviceBuffer(n), DeviceBuffer(8 * n)]
    P.segment_device(tables, bufs[0].ptr, n, bufs[1].ptr, bufs[2].ptr)
    mat, dens = bufs[1].download(np.uint8, n), bufs[2].download(np.float64, n)
    m, d = P.segment(tables, hu)
    np.testing.assert_array_equal(m, mat)
    np.testing.assert_array_equal(d.view(np.uint64), dens.view(np.uint64))
    over = hu.copy()
    N.check(N.lib().dxg_ct_segment(C.byref(tables), N.ptr(over, C.c_double), n, N.ptr(m, C.c_uint8), N.ptr(over, C.c_double)))
    np.testing.assert_array_equal(over.view(np.uint64), dens.view(np.uint64))
    # the materials over the densities: those are written last
    N.check(N.lib().dxg_ct_segment(C.byref(tables), N.ptr(hu, C.c_double), n, N.ptr(d.view(np.uint8), C.c_uint8), N.ptr(d, C.c_double)))
    np.testing.assert_array_equal(d.view(np.uint64), dens.view(np.uint64))
    assert P.last_ms(0) > 0.0


# the 48 MB arrays of 6,000,001 voxels go in chunks, their organ bytes in one piece
@pytest.mark.parametrize("n", [4_500_001, 6_000_001])
def test_dose_table_of_large_host_arrays_equals_resident(n):
    rng = np.random.default_rng(5)
    organ = np.repeat(rng.integers(0, 256, n // 50 + 1, dtype=np.uint8), 50)[:n]
    dose, dens = rng.random(n), rng.uniform(0.0, 2.0, n)
    bufs = [DeviceBuffer.from_array(a) for a in (organ, dose, dens)]
    dev = P.organ_dose_table_device(bufs[0].ptr, bufs[1].ptr, bufs[2].ptr, n, (0.1, 0.1, 0.1))
    np.testing.assert_array_equal(P.organ_dose_table(organ, dose, dens, (0.1, 0.1, 0.1)), dev)


@pytest.mark.parametrize("case", ["held", "segment", "upload", "refused"])
def test_pinned_memory(case):
    """tests/cpp/pinned_memory_check.cpp, whose own hipHostMalloc the library calls."""
    if not build.PINNED_CHECK.exists():
        build.build_pinned_check()
    r = subprocess.run([str(build.PINNED_CHECK), case], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
