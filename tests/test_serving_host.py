"""Host logic of the batch arena and the serving loop (no GPU): slot sizing, HBM budget
admission, FIFO continuous batching, latency percentiles."""
import time

import numpy as np
import pytest

from quick_gpu_cfd_for_neural_network_with_converging_inputs_airfoil2d_version_amd import _native as N
from quick_gpu_cfd_for_neural_network_with_converging_inputs_airfoil2d_version_amd import autotune as AT
from quick_gpu_cfd_for_neural_network_with_converging_inputs_airfoil2d_version_amd import batch as B
from quick_gpu_cfd_for_neural_network_with_converging_inputs_airfoil2d_version_amd import serve as S

from .common import EULER, LAMINAR, case_mesh, merge


def test_slot_capacity_covers_mesh_and_padding():
    _, mesh, _ = case_mesh("G0001", "LF1", LAMINAR)
    for tile in (64, 128, 256):
        cap, feat = B.capacity(mesh, tile)
        info = mesh.info
        assert cap.cells % tile == 0 and cap.cells >= mesh.n_cells + 1 and cap.cells - tile < mesh.n_cells + 1
        assert cap.faces % tile == 0 and cap.faces >= info.n_faces
        assert cap.walls % tile == 0 and cap.walls >= info.n_walls
        assert cap.csr == info.n_cell_faces and cap.terms == info.n_visc_terms
        assert (feat.laminar, feat.sa) == (1, 0)


def test_arena_bytes_monotone_and_budget_inverse():
    _, mesh, _ = case_mesh("G0002", "LF1")
    cap, feat = B.capacity(mesh)
    sizes = [B.arena_bytes([cap] * k, feat, 32) for k in (1, 2, 3, 8, 64)]
    assert all(a < b for a, b in zip(sizes, sizes[1:]))
    assert B.arena_bytes([cap], feat, 64) > B.arena_bytes([cap], feat, 32)
    for k in (1, 7, 40):
        budget = B.arena_bytes([cap] * k, feat, 32)
        assert B.slots_fitting(cap, feat, budget, 32) == k
        assert B.slots_fitting(cap, feat, budget - 1, 32) == k - 1
    # Roughly linear in the slot count: a slot costs the same however many there are.
    per_slot = (sizes[-1] - sizes[0]) / 63
    assert abs(per_slot - (sizes[1] - sizes[0])) < 0.01 * per_slot


def test_envelope_and_union():
    caps, feats = [], []
    for src, ov in (("G0001", LAMINAR), ("G0010", EULER)):
        _, mesh, _ = case_mesh(src, "LF1", ov)
        c, f = B.capacity(mesh)
        caps.append(c)
        feats.append(f)
    env = B.envelope(caps, margin=0.1)
    for name in ("cells", "faces", "walls", "csr", "terms", "groups", "members"):
        assert getattr(env, name) >= max(getattr(c, name) for c in caps) * 1.1 - 1
    assert env.cells % 64 == 0
    u = B.union(feats)
    assert u.laminar == 1 and u.sa == 0


def test_batch_without_device_raises():
    if N.load_library().amr_hip_device_count() > 0:
        pytest.skip("a device is present")
    _, mesh, _ = case_mesh("G0001", "LF1", LAMINAR)
    cap, feat = B.capacity(mesh)
    with pytest.raises(RuntimeError, match="no HIP device"):
        B.Batch.with_slots([cap], feat)


def test_autotuner_few_slot_threshold():
    # two threads per cell must win at every probe up to the threshold (measured shape: they win
    # at 16 running slots and below, lose from 32 up)
    assert AT.choose_few({2: (73.0, 69.0), 8: (85.1, 81.1), 16: (107.0, 102.5), 32: (129.5, 138.4)}) == 16
    assert AT.choose_few({2: (73.0, 75.0), 8: (85.1, 81.1)}) == 0
    assert AT.choose_few({2: (73.0, 70.0), 8: (85.1, 86.0), 16: (107.0, 102.5)}) == 2
    assert AT.choose_few({}) == 0


def test_autotuner_few_slot_shape():
    # The spread that beats the arena's own up to the most slots (the measured shape), or of two alike
    # the faster one.
    assert AT.choose_few_shape({2: {1: 66.2, 2: 61.4, 3: 57.5}, 8: {1: 69.3, 2: 64.5, 3: 72.3},
                                16: {1: 82.6, 2: 77.4, 3: 113.6}, 32: {1: 101.4, 2: 117.1, 3: 166.8}}) == (16, 2)
    assert AT.choose_few_shape({2: {1: 61.0, 2: 55.0, 3: 47.0}, 16: {1: 80.0, 2: 76.0, 3: 79.0}}) == (16, 3)
    assert AT.choose_few_shape({2: {1: 61.0, 2: 55.0, 3: 56.0}, 8: {1: 70.0, 2: 71.0, 3: 65.0}}) == (8, 3)
    assert AT.choose_few_shape({2: {2: 55.0, 3: 56.0}, 8: {2: 71.0, 3: 65.0}}) == (0, 0)
    assert AT.choose_few_shape({}) == (0, 0)


def test_autotuner_keeps_the_larger_tile_within_the_tie_margin():
    # A clear winner is kept whatever its size.
    assert AT.choose({64: 1.00e-3, 128: 1.10e-3, 256: 1.20e-3}) == 64
    assert AT.choose({64: 1.20e-3, 128: 1.00e-3, 256: 1.05e-3}) == 128
    # Within 1% of the fastest the larger tile wins (the measured 256-mesh case: 749.9 / 752.2 us).
    assert AT.choose({64: 749.9e-6, 128: 752.2e-6, 256: 768.2e-6}) == 128
    assert AT.choose({64: 1.000e-3, 128: 1.009e-3, 256: 1.0099e-3}) == 256
    assert AT.choose({64: 1.000e-3, 128: 1.011e-3, 256: 1.02e-3}) == 64
    assert AT.choose({128: 2e-3}) == 128


def test_percentile_and_poisson():
    v = list(range(1, 101))
    assert S.percentile(v, 50) == 50 and S.percentile(v, 99) == 99 and S.percentile(v, 100) == 100
    assert S.percentile([3.0], 99) == 3.0
    t = S.poisson_arrivals(20.0, 20000, seed=1)
    assert np.all(np.diff(t) > 0)
    assert abs(np.mean(np.diff(t)) - 0.05) < 0.002


class FakeMesh:
    def __init__(self, n_cells):
        self.n_cells = n_cells


class FakeBackend:
    """Runs take `duration` seconds of wall time; records concurrency, admission order and slots."""

    def __init__(self, n_slots, max_cells, duration, slot_cells=None):
        self.slot_cells = list(slot_cells) if slot_cells else [max_cells] * n_slots
        self.n_slots, self.duration = len(self.slot_cells), duration
        self.running_runs = {}
        self.peak = 0
        self.started = []
        self.placed = {}

    def fits_slot(self, mesh, slot):
        return mesh.n_cells <= self.slot_cells[slot]

    def slot_size(self, slot):
        return self.slot_cells[slot]

    def fits(self, mesh):
        return any(self.fits_slot(mesh, s) for s in range(self.n_slots))

    def start(self, slot, mesh, params, u0, case, mode, stop_time, budget):
        assert slot not in self.running_runs and self.fits_slot(mesh, slot)
        self.running_runs[slot] = time.perf_counter() + self.duration
        self.started.append(case)
        self.placed[case] = slot
        self.peak = max(self.peak, len(self.running_runs))

    def running(self):
        return len(self.running_runs)

    def poll(self, seconds):
        end = time.perf_counter() + seconds
        while True:
            now = time.perf_counter()
            done = [s for s, t in self.running_runs.items() if t <= now]
            if done or now >= end:
                break
            time.sleep(0.0005)
        out = []
        for s in done:
            del self.running_runs[s]
            out.append((s, {"converged": 1, "steps": 1, "stop_reason": "fake"}))
        return out

    def finish(self, slot):
        assert slot not in self.running_runs


def test_server_fifo_capacity_and_rejection():
    sizes = [100, 100, 500, 100, 100, 100, 100]  # request 2 is too large for a slot
    reqs = [S.Request(i, None, i, arrival=0.002 * i) for i in range(len(sizes))]
    backend = FakeBackend(n_slots=2, max_cells=200, duration=0.03)
    server = S.Server(backend, workers=2, poll_seconds=0.01,
                      mesher=lambda r: (FakeMesh(sizes[r.rid]), None, None))
    rep = server.serve(reqs)
    assert backend.peak == 2
    assert rep["completed"] == 6 and rep["failed"] == 1
    bad = [o for o in rep["outcomes"] if o.error]
    assert bad[0].rid == 2 and "capacity" in bad[0].error
    # First come, first served: admissions follow arrival order (meshing is fast here).
    assert backend.started == [0, 1, 3, 4, 5, 6]
    good = [o for o in rep["outcomes"] if not o.error]
    assert all(o.latency >= 0.03 - 1e-3 for o in good)
    # Three waves of two runs: the last request waits for two runs before it.
    assert rep["p99_latency_seconds"] >= 0.06
    assert 0 < rep["slot_occupancy"] <= 1


def test_server_best_fit_slot_classes():
    # Slots 0-1 hold 100 cells, slot 2 holds 500: small requests take small slots first, a large
    # request waits (first come, first served) until the large slot is free.
    sizes = [90, 400, 80, 450, 70]
    reqs = [S.Request(i, None, i, arrival=0.001 * i) for i in range(len(sizes))]
    backend = FakeBackend(0, 0, duration=0.02, slot_cells=[100, 100, 500])
    server = S.Server(backend, workers=2, poll_seconds=0.005, mesher=lambda r: (FakeMesh(sizes[r.rid]), None, None))
    rep = server.serve(reqs)
    assert rep["completed"] == 5 and rep["failed"] == 0
    assert backend.placed[0] in (0, 1) and backend.placed[1] == 2 and backend.placed[3] == 2
    assert backend.started.index(3) > backend.started.index(1)


def test_mesh_cache_reuses_identical_requests_only():
    from quick_gpu_cfd_for_neural_network_with_converging_inputs_airfoil2d_version_amd import config as CF
    from .common import naca_polygon
    cache = S.MeshCache(capacity=2)
    poly = naca_polygon(0.12)
    a = S.Request(0, poly, CF.make_case("LF1"))
    b = S.Request(1, poly, CF.make_case("LF1"))
    c = S.Request(2, poly, CF.make_case("LF1", {"freestream": {"Mach": 1.3}}))
    m_a, _, u_a = S.build_request_mesh(a, cache)
    m_b, _, u_b = S.build_request_mesh(b, cache)
    m_c, _, u_c = S.build_request_mesh(c, cache)
    assert m_a is m_b and m_c is not m_a
    assert cache.hits == 1 and cache.misses == 2
    assert np.array_equal(u_a, u_b) and not np.array_equal(u_a, u_c)
