"""Batched transport (dxg_batch_*): instances of uneven size in one persistent
launch give exactly what one dxg_transport_run per instance gives (same RNG
streams keyed by seed and history, so identical event counts and scores up to
the order of FP64 atomic additions), on the first (captured) run and on graph
replays."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import opendxmc_amd as dx
from opendxmc_amd import _native as N
from opendxmc_amd import batch_workload as bw


def test_batch_symbols_and_empty_batch():
    b = dx.TransportBatch()
    assert len(b) == 0
    with pytest.raises(N.NativeError) as e:
        b.run()
    assert e.value.code == N.DXG_ERR_STATE


def test_workload_definition():
    inst = bw.instances(8, seed=3, shape_scale=0.25, hist_range=(1e5, 2e5))
    assert len(inst) == 8
    shapes = [ph.dims for ph, _, _ in inst]
    assert shapes[0] == (16, 16, 16) and shapes[1] == (32, 32, 32) and shapes[2] == (24, 40, 20)
    kinds = [type(b).__name__ for _, b, _ in inst]
    assert kinds[0::2] == ["DXBeam"] * 4 and kinds[1::2] == ["CTSequentialBeam"] * 4
    for ph, beam, _ in inst:
        assert 0.05 <= ph.spacing[0] <= 0.2
        assert 0.9e5 <= beam.numberOfParticles() <= 2.1e5


COUNTS = ("histories", "steps", "real_events", "deposits", "uncollided")


@pytest.mark.gpu
def test_batch_equals_one_run_per_instance():
    inst = bw.instances(6, seed=5, shape_scale=0.375, hist_range=(1e5, 6e5))
    single = [bw.make_world(ph) for ph, _, _ in inst]
    batched = [bw.make_world(ph) for ph, _, _ in inst]
    batch = dx.TransportBatch()
    for (ph, beam, s), (world, _) in zip(inst, batched):
        batch.add(world, beam, s)
    assert len(batch) == 6
    for run in range(2):   # the capture, then a graph replay (RNG offsets advance)
        tr = dx.Transport()
        for (ph, beam, s), (world, grid) in zip(inst, single):
            tr.seed = s
            tr(world, beam, None, True)
        ms = batch.run()
        assert ms > 0
        for k, ((_, g1), (_, g2)) in enumerate(zip(single, batched)):
            c1, c2 = g1.counters(), g2.counters()
            for name in COUNTS:
                assert c1[name] == c2[name], (run, k, name, c1[name], c2[name])
            assert g1.histories() == g2.histories()
            e1, e21, n1 = g1.energyScored()
            e2, e22, n2 = g2.energyScored()
            np.testing.assert_array_equal(n1, n2)
            np.testing.assert_allclose(e2, e1, rtol=1e-10, atol=1e-12 * e1.max())
            np.testing.assert_allclose(e22, e21, rtol=1e-10, atol=1e-12 * e21.max())
            assert c2["deposited_energy"] == pytest.approx(c1["deposited_energy"], rel=1e-12)


@pytest.mark.gpu
@pytest.mark.parametrize("copies", [2, 4, 5, 8, 11])
def test_tally_copies_fold_to_the_single_copy(copies, monkeypatch):
    """Worlds with several tally copies (whole and partial groups of four),
    folded by a plain call and by a batch run, against worlds with one; twice,
    so that copies left unzeroed would count again.  A voxel's sums hold the
    same terms in another order: within 2 * events * 2^-53."""
    inst = bw.instances(3, seed=11, shape_scale=0.2, hist_range=(5e4, 2e5))
    monkeypatch.setenv("DXG_TALLY_REPLICAS", "1")
    plain = [bw.make_world(ph) for ph, _, _ in inst]
    monkeypatch.setenv("DXG_TALLY_REPLICAS", str(copies))
    single = [bw.make_world(ph) for ph, _, _ in inst]
    batched = [bw.make_world(ph) for ph, _, _ in inst]
    batch = dx.TransportBatch()
    for (ph, beam, s), (world, _) in zip(inst, batched):
        batch.add(world, beam, s)
    for _ in range(2):
        tr = dx.Transport()
        for worlds in (plain, single):
            for (ph, beam, s), (world, _) in zip(inst, worlds):
                tr.seed = s
                tr(world, beam, None, True)
        batch.run()
        for (_, g0), (_, g1), (_, g2) in zip(plain, single, batched):
            e, e2, ev = g0.energyScored()
            assert ev.sum() > 0
            for g in (g1, g2):
                f, f2, fv = g.energyScored()
                np.testing.assert_array_equal(fv, ev)
                assert np.all(np.abs(f - e) <= 2 * ev * 2.0**-53 * e)
                assert np.all(np.abs(f2 - e2) <= 2 * ev * 2.0**-53 * e2)
                assert all(g.counters()[name] == g0.counters()[name] for name in COUNTS)
