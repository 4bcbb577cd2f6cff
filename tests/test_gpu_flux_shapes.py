"""The spread of the flux launches that an arena chooses by its size (one to three threads per cell)
changes no bit: one mesh as a session (64 cells per tile), in arenas of one slot and of many slots
at the same tile, whose sizes call for three, two and one threads per cell.
"""
import numpy as np
import pytest

from oracle import pyoracle as O
from quick_gpu_cfd_for_neural_network_with_converging_inputs_airfoil2d_version_amd import batch as B
from quick_gpu_cfd_for_neural_network_with_converging_inputs_airfoil2d_version_amd.session import Session

from .common import case_mesh, per_variable_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision, copies", [(64, (1, 8, 16, 28)), (32, (1, 40, 56, 100))])
def test_spread_changes_no_bit(precision, copies):
    # 75 tiles of an LF1 mesh: FP64 arenas hold 2048 waves (27 tiles-of-75 at one thread per cell),
    # FP32 ones 7168.
    case, mesh, params = case_mesh("G0002", "LF1")
    u0 = mesh.initialize(params, case.freestream)
    with Session(mesh, params, u0, precision=precision) as s:
        s.run(60)
        ref = s.download()
    for n in copies:
        print(precision, n, flush=True)
        with B.Batch.of_meshes([mesh] * n, [params] * n, [u0] * n, precision=precision, tile=64) as b:
            b.set_targets(1e30)
            b.run(60)
            for slot in {0, n - 1}:
                np.testing.assert_array_equal(b.download(slot)[0], ref)


@pytest.mark.parametrize("preset", ["LF1", "L7"])  # 75 tiles report to one line, 460 to all
def test_steps_gathered_from_one_line_or_all(preset):
    """The smallest local dt and the arrivals of a slot's blocks: CFL steps with a residual of another
    state and a monitor between them, then fixed steps that are rejected and halved, as the oracle."""
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
