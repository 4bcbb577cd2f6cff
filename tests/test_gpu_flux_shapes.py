"""The spread of the flux launches that an arena chooses by its size (one to three threads per cell)
changes no bit: one mesh as a session (64 cells per tile), in arenas of one slot and of many slots
at the same tile, whose sizes call for three, two and one threads per cell.
"""
import numpy as np
import pytest

from oracle import pyoracle as O
from quick_gpu_cfd_for_neural_network_with_converging_inputs_airfoil2d_version_amd import batch as B
from quick_gpu_cfd_for_neural_network_with_converging_inputs_airfoil2d_version_amd.session import Session

from .common import LAMINAR, case_mesh, merge, per_variable_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision, copies", [(64, {1: 3, 8: 3, 16: 2, 28: 1}), (32, {1: 3, 30: 3, 40: 2, 56: 1, 100: 1})])
def test_spread_changes_no_bit(precision, copies):
    # 75 tiles of an LF1 mesh, one wave each at one thread per cell; the FP64 flux kernels hold 3072
    # waves at a time (13 such meshes at three threads per cell, 20 at two), the FP32 ones 7168 (31, 47).
    case, mesh, params = case_mesh("G0002", "LF1")
    u0 = mesh.initialize(params, case.freestream)
    with Session(mesh, params, u0, precision=precision) as s:
        s.run(60)
        ref = s.download()
    for n, spread in copies.items():
        print(precision, n, flush=True)
        with B.Batch.of_meshes([mesh] * n, [params] * n, [u0] * n, precision=precision, tile=64) as b:
            assert b.launch_shape()[0] == spread
            b.set_targets(1e30)
            b.run(60)
            for slot in {0, n - 1}:
                np.testing.assert_array_equal(b.download(slot)[0], ref)


@pytest.mark.parametrize("preset", ["LF1", "L7"])  # 75 tiles report to one line, 460 to all
def test_steps_gathered_from_one_line_or_all(preset):
    """The smallest local dt and the arrivals of a slot's blocks: CFL steps, then fixed steps that are
    rejected and halved, as the oracle.  (A session's run clears the lines first, so that what a residual
    of another state or a monitor leaves there reaches no step; a batch runs on from them, below.)"""
    case, mesh, params = case_mesh("G0002", preset)
    u0 = mesh.initialize(params, case.freestream)
    ref, meta = O.run(mesh, params, u0, 1e30, maxsteps=8)
    with Session(mesh, params, u0) as s:
        s.run(4)
        s.rhs(ref)
        s.run(2)
        s.monitor(mach=case.mach, aoa=case.aoa)
        s.run(2)
        got = s.download()
    assert s.meta["steps"] == meta["steps"] == 8
    assert abs(s.meta["time"] - meta["time"]) <= 1e-13 * meta["time"]
    assert max(per_variable_l2(got, ref, 5)) <= 1e-10
    params.dt_fixed = 40 * meta["time"] / 8
    ref, meta = O.run(mesh, params, u0, 4.5 * params.dt_fixed)
    with Session(mesh, params, u0) as s:
        s.advance(4.5 * params.dt_fixed)
        got = s.download()
    print(preset, meta["steps"], meta["rejected"], flush=True)
    assert meta["rejected"] > 0 and (s.meta["steps"], s.meta["rejected"]) == (meta["steps"], meta["rejected"])
    assert max(per_variable_l2(got, ref, 5)) <= 1e-10


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("kind", ["sa", "laminar_srd"])
def test_batch_runs_on_after_a_monitor(kind, precision):
    """A monitor between two runs with the same targets leaves its steps in the slots' lines: bitwise the
    run without it, in slots of one line and of all, after an accepted step and in the middle of a
    rejected one."""
    over = None if kind == "sa" else merge(LAMINAR, {"mesh": {"agglomerate_small": False}})
    items = []
    for preset, dt_fixed in (("LF1", 0.0), ("L7", 0.0), ("LF1", 0.0005), ("LF1", 1.0)):
        case, mesh, params = case_mesh("G0002", preset, over) if over else case_mesh("G0002", preset)
        params.dt_fixed = dt_fixed
        items.append((case, mesh, params, mesh.initialize(params, case.freestream)))
    n, frame = len(items), [-1.0, 3.0, -1.0, 1.0, 0.25, 0.0]

    def run(parts, masks):
        with B.Batch.of_meshes([m for _, m, _, _ in items], [p for _, _, p, _ in items], [u for _, _, _, u in items],
                               precision=precision, tile=64) as b:
            b.set_targets(1e30)
            seen = []
            for trials, mask in zip(parts, masks):
                seen.append([(s["steps"], s["rejected"], s["fatal"]) for s in b.run(trials)])
                if mask is not None:
                    _, status = b.monitor(mask, [frame] * n, [c.mach for c, _, _, _ in items], [c.aoa for c, _, _, _ in items])
                    assert [s for s, on in zip(status, mask) if on and s not in (0, 2)] == []
            return seen, [b.download(k) for k in range(n)]

    seen, ref = run([24], [None])
    print(kind, precision, seen, flush=True)
    parts = [1, 2, 1, 20]
    masks = [[1, 1, 1, 1], [1, 0, 1, 1], [0, 1, 1, 1], None]
    seen, got = run(parts, masks)
    print(seen, flush=True)
    assert seen[0][3][:2] == (0, 1)  # the last slot is in the middle of a rejected step at the first monitor
    assert all(steps > 0 for steps, _, _ in seen[-1][:3])
    for k in range(n):
        assert got[k][1] == ref[k][1], k
        np.testing.assert_array_equal(got[k][0], ref[k][0])
